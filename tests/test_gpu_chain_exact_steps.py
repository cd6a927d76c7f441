"""GPU: REFERENCE dot and gemv of entries whose sums pass zero, powers of two and small integers, and of ties, extreme
significands and drifting magnitudes, a wave, a workgroup and a lane per chain, against the oracle's serial order bit for bit."""
import numpy as np
import pytest

from helpers import dev_empty, from_dev, to_dev

pytestmark = pytest.mark.gpu

KINDS = ("signs", "alternating", "twos", "integer", "zeroed", "ties", "extreme", "edges", "drift")
ONE, SIGN = 0x3FFF << 48, 1 << 63


def values(O, kind, seed, n):
    """x and y; "alternating", "twos" and "zeroed" repeat every second element, as a contiguous dot's two chains take every other one."""
    r = np.random.default_rng(seed)
    x, y = np.zeros((n, 2), dtype=np.uint64), np.zeros((n, 2), dtype=np.uint64)
    y[:, 1] = ONE
    sign = r.integers(0, 2, n).astype(np.uint64) << np.uint64(63)
    i = np.arange(n) // 2
    if kind in ("signs", "alternating", "twos"):
        x[:, 1] = ONE
        x[:, 1] |= sign if kind == "signs" else np.where(i & (1 if kind == "alternating" else 2), SIGN, 0).astype(np.uint64)
    elif kind == "integer":
        for v, top in ((x, 8), (y, 4)):
            d = r.integers(-top, top + 1, n).astype(np.float64).view(np.uint64)
            f = d & np.uint64((1 << 52) - 1)
            v[:, 1] = np.where(d << np.uint64(1) == 0, 0, (d & np.uint64(SIGN)) | (((d >> np.uint64(52)) & np.uint64(0x7FF)) + np.uint64(16383 - 1023) << np.uint64(48)) | (f >> np.uint64(4)))
    elif kind == "zeroed":  # x, -x
        x = O.fill(0, seed, n)
        first = np.arange(n) // 4 * 4 + np.arange(n) % 2
        x = x[first]
        x[:, 1] ^= np.where(i & 1, SIGN, 0).astype(np.uint64)
    elif kind == "ties":  # products of 105 bits, a bit below the grid of sums of several units
        for v, drop in ((x, 48), (y, 8)):
            v[:] = O.fill(0, seed + drop, n)
            v[:, 0] &= np.uint64((0xFF << 56) if drop == 8 else 0xF << 60)
            v[:, 1] = (v[:, 1] & np.uint64((1 << 48) - 1)) | ((16383 - r.integers(0, 12, n)).astype(np.uint64) << np.uint64(48)) | (sign if drop == 8 else 0)
    elif kind == "extreme":
        for v in (x, y):
            ones = r.integers(0, 2, (n, 2)).astype(bool)
            v[:, 0] = np.where(ones[:, 0], np.uint64(2**64 - 1), r.integers(0, 2, n).astype(np.uint64))
            v[:, 1] = np.where(ones[:, 1], np.uint64((1 << 48) - 1), np.uint64(0)) | ((16383 + r.integers(-1, 2, n)).astype(np.uint64) << np.uint64(48))
            v[:, 1] |= r.integers(0, 2, n).astype(np.uint64) << np.uint64(63)
    elif kind == "edges":  # sums next to powers of two, with runs of zero products
        x[:, 1] = sign | ((16383 - 20 * r.integers(0, 7, n)).astype(np.uint64) << np.uint64(48)) | np.where(r.integers(0, 2, n) == 1, np.uint64((1 << 48) - 1), np.uint64(0))
        x[:, 0] = np.where(r.integers(0, 2, n) == 1, np.uint64(2**64 - 1), np.uint64(0))
        x[r.integers(0, 3, n) == 0] = 0
    else:
        x, y = O.fill(0, seed, n), O.fill(0, seed + 1, n)
        x[:, 1] += (np.arange(n) // 16 % 40).astype(np.uint64) << np.uint64(48)
    return x, y


def spread(v, inc):
    w = np.zeros(((len(v) - 1) * inc + 1, 2), dtype=np.uint64)
    w[::inc] = v
    return w


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,inc,T", [(700, 1, 1), (333, 2, 1), (9000, 1, 4), (2560, 1, 1), (7001, 2, 2), (70003, 1, 3), (20000, 3, 5)])
def test_dot(O, Q, cuda, kind, n, inc, T):
    print(f"dot {kind} n={n} inc={inc} T={T}", flush=True)
    x, y = (spread(v, inc) for v in values(O, kind, 7 + n, n))
    dx, dy, out = to_dev(x), to_dev(y), dev_empty(1)
    Q.dev_dot(Q.MODE_REFERENCE, n, dx.data_ptr(), inc, dy.data_ptr(), inc, T, out.data_ptr())
    cuda.cuda.synchronize()
    assert np.array_equal(from_dev(out).reshape(2), np.array(O.to_pair(O.dot(n, x, inc, y, inc, T)), dtype=np.uint64))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("layout,m,n,incx", [(0, 13, 900, 1), (0, 9, 333, 2), (1, 21, 500, 1), (1, 3400, 17, 1), (0, 3300, 17, 2)])
def test_gemv(O, Q, cuda, kind, layout, m, n, incx):
    print(f"gemv {kind} layout={layout} {m}x{n} incx={incx}", flush=True)
    a, x = values(O, kind, 9 + n, n)
    A = np.stack([np.roll(a, 4 * i, axis=0) for i in range(m)])
    A = np.ascontiguousarray(A if layout == 0 else A.transpose(1, 0, 2)).reshape(-1, 2)
    lda, x, y = (n if layout == 0 else m), spread(x, incx), O.fill(0, 3, m)
    want = y.copy()
    O.gemv(layout, m, n, 1.0, A, lda, x, incx, 0.0, want, 1)
    dA, dx, dy = to_dev(A), to_dev(x), to_dev(y)
    Q.dev_gemv(Q.MODE_REFERENCE, layout, m, n, 1.0, dA.data_ptr(), lda, dx.data_ptr(), incx, 0.0, dy.data_ptr(), 1)
    cuda.cuda.synchronize()
    assert np.array_equal(from_dev(dy), want)


# more than 4096 chains: rows whose blocks go on failing are left to a kernel of a lane a chain; without scratch, under capture, not
@pytest.mark.parametrize("captured", (False, True))
@pytest.mark.parametrize("layout,m,n,incx", [(0, 2051, 1201, 1), (0, 4099, 600, 2), (1, 4100, 601, 1)])
def test_gemv_rows_left(O, Q, cuda, layout, m, n, incx, captured):
    print(f"rows left layout={layout} {m}x{n} incx={incx} captured={captured}", flush=True)
    A = O.fill(0, 91, m * n).reshape(m, n, 2)
    step = 2 if layout == 0 and incx == 1 else 1  # a contiguous row is two chains
    first = np.arange(n) // (2 * step) * (2 * step) + np.arange(n) % step
    odd = (np.arange(n) // step % 2 == 1) & (first + step < n)
    A[1::3] = A[1::3][:, first]  # every third row: pairs that cancel to far below, from a term on
    A[1::3, :, 1] ^= np.where(odd, SIGN, 0).astype(np.uint64)
    A[2::3, :, 1] &= np.uint64(SIGN | ((1 << 48) - 1))  # subnormal
    A[4::9, : n // 2] = O.fill(0, 92, len(A[4::9]) * (n // 2)).reshape(-1, n // 2, 2)
    x = O.fill(0, 93, n)[first]
    A = np.ascontiguousarray(A if layout == 0 else A.transpose(1, 0, 2)).reshape(-1, 2)
    lda, x, y = (n if layout == 0 else m), spread(x, incx), O.fill(0, 94, m)
    want = y.copy()
    O.gemv(layout, m, n, 1.5, A, lda, x, incx, -0.5, want, 1)
    dA, dx, dy, s = to_dev(A), to_dev(x), to_dev(y), cuda.cuda.Stream()
    cuda.cuda.synchronize()

    def call():
        Q.dev_gemv(Q.MODE_REFERENCE, layout, m, n, 1.5, dA.data_ptr(), lda, dx.data_ptr(), incx, -0.5, dy.data_ptr(), 1, s.cuda_stream)

    for i in range(3):  # the first call makes what a capture of column-major calls needs
        if i == 0 or not captured:
            call()
        else:
            if i == 1:
                g = cuda.cuda.CUDAGraph()
                with cuda.cuda.graph(g, stream=s):
                    call()
            g.replay()
        cuda.cuda.synchronize()
        assert np.array_equal(from_dev(dy), want)
        dy.copy_(to_dev(y))
        cuda.cuda.synchronize()
