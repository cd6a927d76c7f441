"""GPU: the OZAKI batch's slicing of an operand contiguous along k (a wave's tile in LDS) against that of one
contiguous across it: the same problems stored RowMajor and ColMajor, where A and B change places, give the same
C bit for bit.  Sizes around the 8, 16 and 32 elements that the tile is read by, padded leading dimensions."""
import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (1, 5, 7), (31, 33, 8), (32, 32, 9), (33, 31, 15), (5, 70, 16), (70, 5, 17), (64, 64, 31), (65, 63, 32), (40, 40, 33),
        (2, 3, 47), (96, 34, 48), (34, 96, 49), (17, 19, 200)]


@pytest.mark.parametrize("pad", (0, 3))
@pytest.mark.parametrize("kind", (0, 1))
def test_both_layouts_agree(O, Q, cuda, kind, pad):
    print(f"ozaki batch layouts kind={kind} pad={pad}", flush=True)
    results = []
    for layout in (Q.ROW_MAJOR, Q.COL_MAJOR):
        problems, keep = np.zeros(len(DIMS), dtype=Q.GEMM_PROBLEM), []
        for i, (m, n, k) in enumerate(DIMS):
            ptr = []
            for seed, (r, c) in enumerate(((m, k), (k, n), (m, n))):
                v = O.fill(kind, 100 * i + seed, r * c, -30, 30).reshape(r, c, 2)
                if layout == Q.COL_MAJOR:
                    v = v.transpose(1, 0, 2)
                w = np.zeros((v.shape[0], v.shape[1] + pad, 2), dtype=np.uint64)
                w[:, : v.shape[1]] = v
                keep.append(to_dev(w.reshape(-1, 2)))
                ptr.append((keep[-1], v.shape[1], v.shape[1] + pad))
            p = problems[i]
            p["m"], p["n"], p["k"] = m, n, k
            p["A"], p["B"], p["C"] = (t.data_ptr() for t, _, _ in ptr)
            p["lda"], p["ldb"], p["ldc"] = (ld for _, _, ld in ptr)
            problems["alpha"][i], problems["beta"][i] = Q.from_double(1.5), Q.from_double(-0.5)
        d = cuda.from_numpy(problems.view(np.uint8).copy()).cuda()
        Q.dev_gemm_batched(Q.MODE_OZAKI, layout, len(DIMS), d.data_ptr())
        cuda.cuda.synchronize()
        out = []
        for i, (m, n, k) in enumerate(DIMS):
            rows, cols = (m, n) if layout == Q.ROW_MAJOR else (n, m)
            c = np.array(from_dev(keep[3 * i + 2])).reshape(rows, cols + pad, 2)[:, :cols]
            out.append(c if layout == Q.ROW_MAJOR else c.transpose(1, 0, 2))
        results.append(out)
    for dims, a, b in zip(DIMS, *results):
        assert np.array_equal(a, b), dims
