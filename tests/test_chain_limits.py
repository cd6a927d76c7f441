"""The accumulating FMA chain (qblas_amd/csrc/chain.hpp) at the limits of its fast step and on operands with many zeros, compiled for
the host: bit for bit the packed fma_packed after every step."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chain_at_its_limits(tmp_path):
    exe = tmp_path / "chain_limits_host_check"
    src = os.path.join(ROOT, "tests", "cpu", "chain_limits_host_check.cpp")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-Wno-unknown-pragmas", "-o", str(exe), src], check=True)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "2000"], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:]
        lines = [line.split() for line in r.stdout.splitlines()]
        assert len(lines) == 7 and all(line[-1] == "0" for line in lines)
        # the fast step takes part: its limits are inside the ranges
        assert all(0 < int(line[4]) < int(line[2]) for line in lines)
