"""GPU: REFERENCE gemm, gemv (a lane a chain) and batches of matrices with many zeros of both signs, an infinity and a subnormal
among them, against the oracle's serial order, bit for bit (NaN as one)."""
import numpy as np
import pytest

from helpers import from_dev, to_dev
from test_gpu_chain_scan import plain

pytestmark = pytest.mark.gpu


def values(O, seed, n, zeros, special):
    v, r = O.fill(0, seed, n), np.random.default_rng(seed)
    v[r.random(n) < zeros] = 0
    v[r.random(n) < zeros / 3] = (0, 1 << 63)
    if special:
        v[n // 2], v[n // 3] = (0, 0x7FFF << 48), (12345, 1 << 40)
    return v


@pytest.mark.parametrize("special", (False, True))
@pytest.mark.parametrize("zeros", (0.5, 0.9, 1.0))
@pytest.mark.parametrize("layout,m,n,k", [(0, 33, 40, 130), (1, 17, 31, 64), (0, 70, 65, 300)])
def test_gemm(O, Q, cuda, layout, m, n, k, zeros, special):
    print(f"gemm layout={layout} {m}x{n}x{k} zeros={zeros} special={special}", flush=True)
    A, B, C = values(O, 1, m * k, zeros, special), values(O, 2, k * n, zeros, False), values(O, 3, m * n, zeros, False)
    lda, ldb, ldc = (k, n, n) if layout == 0 else (m, k, m)
    for alpha, beta in ((1.5, -0.5), (-1.0, 0.0)):
        want = C.copy()
        O.gemm(layout, m, n, k, alpha, A, lda, B, ldb, beta, want, ldc)
        dA, dB, dC = to_dev(A), to_dev(B), to_dev(C)
        Q.dev_gemm(Q.MODE_REFERENCE, layout, m, n, k, alpha, dA.data_ptr(), lda, dB.data_ptr(), ldb, beta, dC.data_ptr(), ldc)
        dE = to_dev(C)
        p = np.zeros(1, dtype=Q.GEMM_PROBLEM)
        p["m"], p["n"], p["k"], p["lda"], p["ldb"], p["ldc"] = m, n, k, lda, ldb, ldc
        p["A"], p["B"], p["C"] = dA.data_ptr(), dB.data_ptr(), dE.data_ptr()
        p["alpha"][0], p["beta"][0] = Q.from_double(alpha), Q.from_double(beta)
        dp = cuda.from_numpy(p.view(np.uint8).copy()).to("cuda")
        Q.dev_gemm_batched(Q.MODE_REFERENCE, layout, 1, dp.data_ptr())
        cuda.cuda.synchronize()
        assert np.array_equal(plain(from_dev(dC)), plain(want))
        assert np.array_equal(plain(from_dev(dE)), plain(want))


@pytest.mark.parametrize("special", (False, True))
@pytest.mark.parametrize("zeros", (0.5, 0.9, 1.0))
@pytest.mark.parametrize("layout,m,n,incx", [(0, 6500, 35, 1), (0, 13000, 33, 2), (1, 13000, 37, 1)])
def test_gemv_lane_per_chain(O, Q, cuda, layout, m, n, incx, zeros, special):
    print(f"gemv layout={layout} {m}x{n} zeros={zeros} special={special}", flush=True)
    lda = n if layout == 0 else m
    A, x, y = values(O, 4, m * n, zeros, special), values(O, 5, (n - 1) * incx + 1, zeros, False), values(O, 6, m, zeros, False)
    want = y.copy()
    O.gemv(layout, m, n, 1.5, A, lda, x, incx, -0.5, want, 1)
    dA, dx, dy = to_dev(A), to_dev(x), to_dev(y)
    Q.dev_gemv(Q.MODE_REFERENCE, layout, m, n, 1.5, dA.data_ptr(), lda, dx.data_ptr(), incx, -0.5, dy.data_ptr(), 1)
    cuda.cuda.synchronize()
    assert np.array_equal(plain(from_dev(dy)), plain(want))
