"""GPU: the EXACT dot that one workgroup finishes by itself (n <= 8192), and the first size above it, against
the oracle's correctly rounded sum: fewer elements than the workgroup has lanes, one to sixteen a lane, strides,
exact cancellation, and products far apart (the full-range path)."""
import numpy as np
import pytest

from helpers import dev_empty, from_dev, pair, to_dev

pytestmark = pytest.mark.gpu


def values(O, kind, seed, n):
    if kind == "far":
        return O.fill(1, seed, n, -6000, 6000), O.fill(1, seed + 1, n, -6000, 6000)
    if kind == "log":
        return O.fill(1, seed, n, -30, 30), O.fill(1, seed + 1, n, -30, 30)
    if kind == "cancel":
        return O.fill(2, seed, n), O.fill_pair_y(seed, n)
    x, y = O.fill(0, seed, n), O.fill(0, seed + 1, n)
    if kind == "zero":  # pairs that cancel exactly, and an element of zero
        x[1::2], y[1::2] = x[0 : n - n % 2 : 2], y[0 : n - n % 2 : 2]
        x[1::2, 1] ^= np.uint64(1 << 63)
        x[n - n % 2 :] = 0
    return x, y


@pytest.mark.parametrize("kind", ("uniform", "log", "cancel", "zero", "far"))
@pytest.mark.parametrize("n,incx,incy", [(1, 1, 1), (65, 1, 1), (511, 1, 1), (512, 1, 1), (513, 2, 1), (1001, 1, 1), (1025, 1, 3),
                                         (1537, 1, 1), (2048, 1, 1), (2049, 2, 1), (8191, 1, 1), (8192, 1, 2), (8193, 1, 1)])
def test_dot_exact_small(O, Q, cuda, n, incx, incy, kind):
    print(f"dot exact {kind} n={n} incx={incx} incy={incy}", flush=True)
    u, v = values(O, kind, 71 + n, n)
    x, y = np.zeros(((n - 1) * incx + 1, 2), dtype=np.uint64), np.zeros(((n - 1) * incy + 1, 2), dtype=np.uint64)
    x[::incx], y[::incy] = u, v
    dx, dy, out = to_dev(x), to_dev(y), dev_empty(1)
    for _ in range(2):  # the second call finds the first one's header
        Q.dev_dot(Q.MODE_EXACT, n, dx.data_ptr(), incx, dy.data_ptr(), incy, 1, out.data_ptr())
        cuda.cuda.synchronize()
        assert Q.dev_exact_status() == 0
        assert pair(from_dev(out)[0]) == O.exact_dot(u, v)[0]


@pytest.mark.parametrize("n", (3, 600, 8192))
def test_dot_exact_small_specials(O, Q, cuda, n):
    print(f"dot exact specials n={n}", flush=True)
    inf = (0, 0x7FFF << 48)
    for at, x0, y0, want in (((n - 1,), inf, (0, 0x3FFF << 48), inf), ((0,), inf, (0, 0xBFFF << 48), (0, 0xFFFF << 48)),
                             ((n // 2,), inf, (0, 0), None), ((0, n - 1), None, None, None)):
        x, y = O.fill(0, 5, n), O.fill(0, 6, n)
        if x0 is None:  # infinities of both signs
            x[0], y[0], x[n - 1], y[n - 1] = inf, (0, 0x3FFF << 48), inf, (0, 0xBFFF << 48)
        else:
            x[at[0]], y[at[0]] = x0, y0
        dx, dy, out = to_dev(x), to_dev(y), dev_empty(1)
        Q.dev_dot(Q.MODE_EXACT, n, dx.data_ptr(), 1, dy.data_ptr(), 1, 1, out.data_ptr())
        cuda.cuda.synchronize()
        got = pair(from_dev(out)[0])
        if want is None:
            assert (got[1] >> 48) & 0x7FFF == 0x7FFF and (got[0] or got[1] & ((1 << 48) - 1))
        else:
            assert got == want
