"""Both forms of the scanned FMA chain (qblas_amd/csrc/chain_scan.hpp), a wave's and a workgroup's, compiled for the host: bit for
bit the serial packed fma, and on entries whose sums pass zero, powers of two and small integers no more passes than on others."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_scanned_chains(tmp_path):
    exe = tmp_path / "chain_group_host_check"
    src = os.path.join(ROOT, "tests", "cpu", "chain_group_host_check.cpp")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-Wno-unknown-pragmas", "-o", str(exe), src], check=True)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "200"], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:]
        lines = [line.split() for line in r.stdout.splitlines()]
        assert len(lines) == 23 and all(line[-1] == "0" for line in lines)
        for line in lines:
            steps, passes, alone, _, left, group_steps, group_passes = (int(line[i]) for i in (2, 4, 6, 8, 10, 13, 15))
            kind = line[0][:-1]
            if kind in ("uniform", "wide", "double", "positive", "sparse", "ties"):  # get on by themselves
                assert alone < steps / 100 and left == 0, line
            if kind in ("uniform", "double", "positive", "ties", "ones", "signs", "alternating", "twos", "integer", "difference", "zeroed", "brink"):
                # 150 chains of a wave, 64 steps a pass; 50 of a workgroup, 2048 steps; and some passes of each to find out
                assert passes < 1.5 * steps / 64 + 150 * 12 and left == 0, line
                assert group_passes < 2 * group_steps / 2048 + 50 * 6, line
