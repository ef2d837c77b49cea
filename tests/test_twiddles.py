"""Roots of unity as products of two (no GPU), as the plans' tables hold them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++"


def test_split_roots(tmp_path):
    exe = str(tmp_path / "split_roots_host")
    subprocess.run([CXX, "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(ROOT, "tests/c_abi/split_roots_host.cpp"),
                    os.path.join(ROOT, "perf-libs-fft_amd/csrc/twiddles.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout) > 10 ** 6, r.stdout
