"""Host check of the flexible chains (no GPU): every chain the planner can
choose addresses its LDS as the Stockham definition says."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_flex_chains_address_every_element(tmp_path):
    exe = str(tmp_path / "flex_chain_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-o", exe,
                    os.path.join(ROOT, "tests/c_abi/flex_chain_host.cpp"),
                    os.path.join(ROOT, "perf-libs-fft_amd/csrc/flex_chain.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 1500
