"""Flexible chains of small batches of real transforms (no GPU): every chain
addresses its LDS as the Stockham definition says, and members get the threads
that the loads and stores around the chain need."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_waiting_chains(tmp_path):
    exe = str(tmp_path / "flex_wait_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-o", exe,
                    os.path.join(ROOT, "tests/c_abi/flex_wait_host.cpp"),
                    os.path.join(ROOT, "perf-libs-fft_amd/csrc/flex_chain.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    count, more = (int(w) for w in r.stdout.split() if w.isdigit())
    assert more > 0.8 * count / 12
