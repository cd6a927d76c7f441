"""The OZAKI finishes' epilogue (qblas_amd/csrc/finish_top.hpp), compiled for the host: the result and the bound of
finish_reg_top, bit for bit, on random, short, cancelling, special and extreme operands."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_finish_top_matches_finish_reg_top(tmp_path):
    exe = tmp_path / "finish_top_host_check"
    src = os.path.join(ROOT, "tests", "cpu", "finish_top_host_check.cpp")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-Wno-unknown-pragmas", "-o", str(exe), src], check=True)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "100000"], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:]
        assert r.stdout.count("mismatches 0") == 3
