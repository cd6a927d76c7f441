"""GPU: the REFERENCE dot and gemv by a wave per chain (64 steps at a time) against the oracle's serial
order, bit for bit: chain lengths around a block of 64, operands that leave the block's fast path
(zeros, subnormals, infinities, NaN, large cancelling pairs, ties, sums next to powers of two), and
sizes on both sides of the rule that chooses between a wave and a lane per chain."""
import numpy as np
import pytest

from helpers import dev_empty, from_dev, to_dev

pytestmark = pytest.mark.gpu

KINDS = ("uniform", "wide", "cancel", "double", "sparse", "ones", "subnormal", "inf", "nan", "overflow")


def values(O, kind, seed, n, second=False):
    if kind in ("uniform", "wide"):
        return O.fill(0 if kind == "uniform" else 1, seed, n, -30, 30)
    if kind == "cancel":
        return O.fill_pair_y(seed, n) if second else O.fill(2, seed, n)
    v = O.fill(0, seed + second, n)
    r = np.random.default_rng(seed + second)
    if kind == "double":
        v[:, 0] &= np.uint64(0xF << 60)
    elif kind == "sparse":
        v[r.random(n) < 0.6] = 0
        v[r.random(n) < 0.1] = (0, 1 << 63)
    elif kind == "ones":
        v[:] = (0, 0x3FFF << 48)
    elif kind == "subnormal":
        v[r.random(n) < 0.05, 1] &= np.uint64((1 << 63) | ((1 << 48) - 1))
    elif kind in ("inf", "nan"):
        v[(3 * n) // 4, :] = (0, 0x7FFF << 48)
        if kind == "nan":
            v[(4 * n) // 5, :] = (0, (0x7FFF << 48) | (1 << 47))
    elif kind == "overflow":
        v[:, 1] += np.uint64(0x1FF0 << 48) if n < 5 or not second else np.uint64(0x1FF8 << 48)
    return v


def plain(a):
    """The words, every NaN as one."""
    a = np.array(a, dtype=np.uint64).reshape(-1, 2)
    nan = (((a[:, 1] >> np.uint64(48)) & np.uint64(0x7FFF)) == 0x7FFF) & (((a[:, 1] << np.uint64(16)) | a[:, 0]) != 0)
    a[nan] = (0, 0x7FFF8 << 44)
    return a


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,inc,T", [(1, 1, 1), (127, 1, 1), (128, 1, 1), (129, 1, 1), (131, 1, 1), (65, 2, 1), (64, 3, 1),
                                     (1003, 1, 4), (640, 2, 5), (6001, 1, 70)])
def test_dot(O, Q, cuda, kind, n, inc, T):
    print(f"dot {kind} n={n} inc={inc} T={T}", flush=True)
    size = (n - 1) * inc + 1
    x, y = values(O, kind, 11 + n, size), values(O, kind, 11 + n, size, True)
    dx, dy, out = to_dev(x), to_dev(y), dev_empty(1)
    Q.dev_dot(Q.MODE_REFERENCE, n, dx.data_ptr(), inc, dy.data_ptr(), inc, T, out.data_ptr())
    cuda.cuda.synchronize()
    assert np.array_equal(plain(from_dev(out)), plain(O.to_pair(O.dot(n, x, inc, y, inc, T))))


# chains of a workgroup each: 1280 steps are the fewest, 2048 are done at a time; 256 chains are the most
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,inc,T", [(1279, 2, 1), (1280, 2, 1), (2112, 3, 1), (2113, 2, 1), (2560, 1, 1), (4225, 1, 1), (8323, 1, 2), (21503, 2, 5),
                                     (66000, 1, 3), (327685, 1, 128), (327697, 2, 256)])
def test_dot_workgroup_per_chain(O, Q, cuda, kind, n, inc, T):
    test_dot(O, Q, cuda, kind, n, inc, T)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("layout,m,n,incx", [(0, 3, 129, 1), (0, 5, 64, 2), (0, 7, 1001, 1), (1, 9, 65, 1), (1, 17, 1000, 2), (1, 8, 63, 1)])
def test_gemv(O, Q, cuda, kind, layout, m, n, incx):
    print(f"gemv {kind} layout={layout} {m}x{n} incx={incx}", flush=True)
    lda = (n if layout == 0 else m) + 1
    A = values(O, kind, 21 + n, (m if layout == 0 else n) * lda)
    x = values(O, kind, 21 + n, (n - 1) * incx + 1, True)
    y = values(O, "uniform", 22, m)
    y[0] = (0, 1 << 63)
    for alpha, beta in ((1.0, 0.0), (1.5, -0.5)):
        want = y.copy()
        O.gemv(layout, m, n, alpha, A, lda, x, incx, beta, want, 1)
        dA, dx, dy = to_dev(A), to_dev(x), to_dev(y)
        Q.dev_gemv(Q.MODE_REFERENCE, layout, m, n, alpha, dA.data_ptr(), lda, dx.data_ptr(), incx, beta, dy.data_ptr(), 1)
        cuda.cuda.synchronize()
        assert np.array_equal(plain(from_dev(dy)), plain(want))


# chains (64 ceil(len / 64) + 128) <= 36864 len: 3072 chains of 16 are the last that get a wave each
@pytest.mark.parametrize("layout,m,n,incx", [(1, 3072, 16, 1), (1, 3073, 16, 1), (0, 3072, 16, 2), (0, 3073, 16, 2),
                                             (0, 1536, 32, 1), (0, 1537, 33, 1), (0, 5000, 45, 1), (1, 3075, 33, 2)])
def test_gemv_either_side_of_the_rule(O, Q, cuda, layout, m, n, incx):
    print(f"gemv layout={layout} {m}x{n} incx={incx}", flush=True)
    lda = n if layout == 0 else m
    A, x, y = O.fill(0, 31, m * n), O.fill(0, 32, (n - 1) * incx + 1), O.fill(0, 33, m)
    want = y.copy()
    O.gemv(layout, m, n, 1.5, A, lda, x, incx, -0.5, want, 1)
    dA, dx, dy = to_dev(A), to_dev(x), to_dev(y)
    Q.dev_gemv(Q.MODE_REFERENCE, layout, m, n, 1.5, dA.data_ptr(), lda, dx.data_ptr(), incx, -0.5, dy.data_ptr(), 1)
    cuda.cuda.synchronize()
    assert np.array_equal(from_dev(dy), want)


@pytest.mark.parametrize("kind", ("cancel", "sparse", "subnormal", "nan"))
@pytest.mark.parametrize("layout,m,n,incx", [(0, 1600, 31, 1), (0, 3300, 17, 2), (1, 3200, 15, 1)])
def test_gemv_lane_per_chain(O, Q, cuda, kind, layout, m, n, incx):
    test_gemv(O, Q, cuda, kind, layout, m, n, incx)
