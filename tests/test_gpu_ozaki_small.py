"""GPU: the OZAKI gemm's small-product launches (one scaling kernel for both operands, halves of residue fragments, row
quarters of reconstruction blocks) on both sides of their limits, both layouts: sampled entries within 2^-104 of the exact
value, and a small product bit-identical to the same rows and columns inside a product that takes the other launches."""
import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -104


def gemm(Q, cuda, layout, m, n, k, alpha, beta, A, B, C, t):
    Q.set_ozaki_method(Q.OZAKI_CRT)
    Q.set_ozaki_crt_bits(t)
    lda, ldb, ldc = (k, n, n) if layout == 0 else (m, k, m)
    try:
        dA, dB, dC = to_dev(A), to_dev(B), to_dev(C)
        Q.dev_gemm(Q.MODE_OZAKI, layout, m, n, k, alpha, dA.data_ptr(), lda, dB.data_ptr(), ldb, beta, dC.data_ptr(), ldc)
        cuda.cuda.synchronize()
        assert Q.dev_exact_status() == 0
    finally:
        Q.set_ozaki_crt_bits(0)
        Q.set_ozaki_method(Q.OZAKI_AUTO)
    return from_dev(dC)


# scaling: 4096 rows and 1024 columns are the last of the small kernel; halves up to 1536 fragment positions of both
# operands ((m + n) / 32 row blocks, padded to 256 rows, times k / 32); row quarters up to 512 blocks
@pytest.mark.parametrize("layout,m,n,k,alpha,beta", [
    (0, 1, 1, 1, 1.0, 0.0), (1, 15, 17, 65, 1.5, -0.5), (0, 300, 40, 1024, 1.0, 0.0), (1, 300, 40, 1025, -1.0, 0.0),
    (0, 4096, 5, 33, 1.0, 0.0), (1, 4097, 5, 33, 1.5, 1.0), (1, 3, 4097, 70, 1.0, 0.0),
    (0, 250, 250, 96 * 32, 1.0, 0.0), (1, 250, 250, 97 * 32, 1.0, 0.0),
    (0, 512, 1024, 40, 1.0, 0.0), (1, 513, 1024, 40, 1.5, -0.5)])
def test_either_side_of_the_limits(O, Q, cuda, layout, m, n, k, alpha, beta):
    print(f"ozaki layout={layout} {m}x{n}x{k}", flush=True)
    A, B, C = O.fill(1, 71, m * k, -10, 10), O.fill(1, 72, k * n, -10, 10), O.fill(0, 73, m * n)
    got = gemm(Q, cuda, layout, m, n, k, alpha, beta, A, B, C, 130)
    r = np.random.default_rng(7)
    ii, jj = r.integers(0, m, 400), r.integers(0, n, 400)
    st = lambda rows, cols: (cols, 1) if layout == 0 else (1, rows)
    cs = st(m, n)
    cand = np.ascontiguousarray(got[ii * cs[0] + jj * cs[1]])
    _, rel = O.exact_gemm_samples(ii, jj, k, alpha, A, st(m, k), B, st(k, n), beta, C, cs, cand=cand)
    assert float(np.max(rel)) <= TOL


def test_small_equals_part_of_large(O, Q, cuda):
    m, n, k, M, N = 40, 50, 60, 1100, 1000  # the large one: 1100 x 1000, whole blocks, whole fragments
    A, B = O.fill(1, 81, M * k, -10, 10), O.fill(1, 82, k * N, -10, 10)
    A[3 * k:4 * k] = 0                       # a zero row and a row with an infinity
    A[5 * k + 7] = (0, 0x7FFF << 48)
    big = gemm(Q, cuda, 0, M, N, k, 1.0, 0.0, A, B, np.zeros((M * N, 2), dtype=np.uint64), 120).reshape(M, N, 2)
    part = gemm(Q, cuda, 0, m, n, k, 1.0, 0.0, np.ascontiguousarray(A[:m * k]), np.ascontiguousarray(B.reshape(k, N, 2)[:, :n].reshape(-1, 2)),
                np.zeros((m * n, 2), dtype=np.uint64), 120).reshape(m, n, 2)
    assert np.array_equal(part, big[:m, :n])
