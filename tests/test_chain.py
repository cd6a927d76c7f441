"""The accumulating FMA chain of the REFERENCE-order kernels (qblas_amd/csrc/chain.hpp), compiled for
the host: bit for bit the packed fma_packed after every step, over uniform, log-uniform, short,
cancelling, extreme-significand, special, subnormal and overflowing operands."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chain_matches_packed_fma(tmp_path):
    exe = tmp_path / "chain_host_check"
    src = os.path.join(ROOT, "tests", "cpu", "chain_host_check.cpp")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-Wno-unknown-pragmas", "-o", str(exe), src], check=True)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "3000"], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:]
        lines = r.stdout.splitlines()
        assert len(lines) == 11 and all(line.endswith("mismatches 0") for line in lines)
        # the fast step takes what the benchmark data brings
        steps = {line.split(":")[0]: (int(line.split()[2]), int(line.split()[4])) for line in lines}
        assert all(steps[kind][1] * 100 < steps[kind][0] for kind in ("uniform", "wide", "double", "short"))


def test_wave_chain_matches_packed_fma(tmp_path):
    """The wave-wide chain (qblas_amd/csrc/chain_scan.hpp), its lanes as loops: whole chains, and few steps by themselves."""
    exe = tmp_path / "chain_scan_host_check"
    src = os.path.join(ROOT, "tests", "cpu", "chain_scan_host_check.cpp")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-Wno-unknown-pragmas", "-o", str(exe), src], check=True)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "600"], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:]
        lines = r.stdout.splitlines()
        assert len(lines) == 14 and all(line.endswith("wrong chains 0") for line in lines)
        single = {line.split(":")[0]: int(line.split()[8]) / int(line.split()[2]) for line in lines}
        assert all(single[kind] < 0.01 for kind in ("uniform", "wide", "double", "sparse"))
