"""GPU: the scratch of the REFERENCE gemm: calls return while the device is busy, on more streams than have scratch and where a
larger call outgrows a stream's; results on all of them against the oracle bit for bit; a thread that ends gives
its memory back."""
import threading

import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def product(O, m, n, k, seed):
    A, B, C = O.fill(0, seed, m * k), O.fill(0, seed + 1, k * n), O.fill(0, seed + 2, m * n)
    want = C.copy()
    O.gemm(0, m, n, k, 1.5, A, k, B, n, -0.5, want, n)
    return (m, n, k), to_dev(A), to_dev(B), to_dev(C), want


def call(Q, p, stream):
    (m, n, k), A, B, C, _ = p
    Q.dev_gemm(Q.MODE_REFERENCE, 0, m, n, k, 1.5, A.data_ptr(), k, B.data_ptr(), n, -0.5, C.data_ptr(), n, stream.cuda_stream)


def test_calls_do_not_wait(O, Q, cuda):
    failed = []

    def body():  # a new thread has no scratch
        try:
            small = [product(O, 40, 50, 300, 100 + 3 * i) for i in range(6)]
            large = [product(O, 90, 70, 800, 200 + 3 * i) for i in range(6)]
            streams = [cuda.cuda.Stream() for _ in range(6)]
            for s, p in zip(streams, small):
                call(Q, p, s)
            cuda.cuda.synchronize()
            held = [cuda.cuda.Stream(), streams[0]]
            done = []
            for s in held:
                with cuda.cuda.stream(s):
                    cuda.cuda._sleep(100_000_000)
                    done.append(cuda.cuda.Event())
                    done[-1].record(s)
            print("calls on six streams beside busy ones", flush=True)
            for s, p in zip(streams, large):
                call(Q, p, s)
            assert not any(e.query() for e in done)
            cuda.cuda.synchronize()
            for p in small + large:
                assert np.array_equal(from_dev(p[3]), p[4])
        except BaseException as e:
            failed.append(e)

    t = threading.Thread(target=body)
    t.start()
    t.join()
    assert not failed, failed


def test_a_thread_gives_its_scratch_back(O, Q, cuda):
    p = product(O, 700, 690, 126 * 8, 300)  # 62 MB of scratch
    free = []
    for i in range(5):
        print(f"thread {i}", flush=True)
        t = threading.Thread(target=lambda: (call(Q, p, cuda.cuda.current_stream()), cuda.cuda.synchronize()))
        t.start()
        t.join()
        free.append(cuda.cuda.mem_get_info()[0])
    assert free[0] - free[-1] < 32 << 20
