"""GPU: the REFERENCE gemm with its blocks of k over workgroups, and without, against the oracle bit for bit: one block and a
short one, both sides of the tile count that decides, more blocks than one round of the workspace holds, and a capture
that has no workspace."""
import threading

import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,m,n,k,alpha,beta,kind", [
    (0, 17, 33, 127, 1.5, -0.5, 0), (1, 1, 1, 253, 1.0, 0.0, 0), (0, 65, 16, 126, -0.75, 1.0, 1), (1, 70, 90, 1009, 1.5, 0.25, 1),
    (0, 700, 690, 126 * 9 + 5, 1.5, -0.5, 0),   # 7.7 MB a block: 8 blocks a round
    (1, 720, 720, 130, 1.0, 1.0, 0), (0, 730, 730, 130, 1.0, 1.0, 0),   # 2025 tiles and 2116
])
def test_gemm_blocks_of_k(O, Q, cuda, layout, m, n, k, alpha, beta, kind):
    print(f"gemm layout={layout} {m}x{n}x{k} kind={kind}", flush=True)
    lda, ldb, ldc = (k, n, n) if layout == 0 else (m, k, m)
    A, B, C = O.fill(kind, 51, m * k, -30, 30), O.fill(kind, 52, k * n, -30, 30), O.fill(0, 53, m * n)
    C[0] = (0, 1 << 63)
    want = C.copy()
    O.gemm(layout, m, n, k, alpha, A, lda, B, ldb, beta, want, ldc)
    dA, dB, dC = to_dev(A), to_dev(B), to_dev(C)
    Q.dev_gemm(Q.MODE_REFERENCE, layout, m, n, k, alpha, dA.data_ptr(), lda, dB.data_ptr(), ldb, beta, dC.data_ptr(), ldc)
    cuda.cuda.synchronize()
    assert np.array_equal(from_dev(dC), want)


# 35 x 36 = 1260 tiles stage 32 values of k at a time, 36 x 36 = 1296 sixteen; 127 is two blocks of k
@pytest.mark.parametrize("kind", (0, 1))
@pytest.mark.parametrize("layout,m,n,k", [(0, 560, 561, 33), (0, 561, 576, 15), (1, 576, 561, 16), (0, 562, 563, 33), (1, 561, 575, 127), (1, 560, 575, 127)])
def test_gemm_either_side_of_the_staging_rule(O, Q, cuda, layout, m, n, k, kind):
    test_gemm_blocks_of_k(O, Q, cuda, layout, m, n, k, 1.5, -0.5, kind)


def test_gemm_captured_without_a_workspace(O, Q, cuda):
    m, n, k = 40, 50, 400
    A, B, C = O.fill(0, 61, m * k), O.fill(0, 62, k * n), O.fill(0, 63, m * n)
    want = C.copy()
    O.gemm(0, m, n, k, 1.5, A, k, B, n, 0.0, want, n)
    dA, dB, dC = to_dev(A), to_dev(B), to_dev(C)
    failed = []

    def capture():  # a new thread has no workspaces
        try:
            s = cuda.cuda.Stream()
            g = cuda.cuda.CUDAGraph()
            with cuda.cuda.graph(g, stream=s):
                Q.dev_gemm(Q.MODE_REFERENCE, 0, m, n, k, 1.5, dA.data_ptr(), k, dB.data_ptr(), n, 0.0, dC.data_ptr(), n,
                           cuda.cuda.current_stream().cuda_stream)
            for _ in range(3):
                dC.zero_()
                g.replay()
                cuda.cuda.synchronize()
                assert np.array_equal(from_dev(dC), want)
        except BaseException as e:
            failed.append(e)

    t = threading.Thread(target=capture)
    t.start()
    t.join()
    assert not failed, failed
