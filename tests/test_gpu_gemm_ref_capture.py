"""GPU: the REFERENCE gemm under capture after eager calls of the same thread and stream, whose scratch a graph may not use: two
forked branches of one capture, two graphs captured on one stream and replayed on two, and replays beside eager calls on
the stream of the capture, each C against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

SHAPE = (40, 50, 1400)  # 12 blocks of k


class Product:
    def __init__(self, O, Q, cuda, seed):
        m, n, k = SHAPE
        A, B, C = O.fill(0, seed, m * k), O.fill(0, seed + 1, k * n), O.fill(0, seed + 2, m * n)
        self.Q, self.cuda, self.want = Q, cuda, C.copy()
        O.gemm(0, m, n, k, 1.5, A, k, B, n, 0.0, self.want, n)
        self.A, self.B, self.C = to_dev(A), to_dev(B), to_dev(C)

    def run(self, stream):
        m, n, k = SHAPE
        self.Q.dev_gemm(self.Q.MODE_REFERENCE, 0, m, n, k, 1.5, self.A.data_ptr(), k, self.B.data_ptr(), n, 0.0,
                        self.C.data_ptr(), n, stream.cuda_stream)

    def check(self):
        assert np.array_equal(from_dev(self.C), self.want)
        self.C.zero_()


@pytest.fixture
def work(O, Q, cuda):
    p = [Product(O, Q, cuda, 71 + 3 * i) for i in range(3)]
    s = [cuda.cuda.Stream(), cuda.cuda.Stream()]
    cuda.cuda.synchronize()
    p[0].run(s[0])  # the stream has its scratch now
    cuda.cuda.synchronize()
    p[0].check()
    cuda.cuda.synchronize()
    return p, s


def capture(cuda, stream, body):
    g = cuda.cuda.CUDAGraph()
    with cuda.cuda.graph(g, stream=stream):
        body()
    return g


def test_forked_branches(cuda, work):
    p, s = work

    def body():
        s[1].wait_stream(s[0])
        p[0].run(s[0])
        p[1].run(s[1])
        s[0].wait_stream(s[1])

    g = capture(cuda, s[0], body)
    for i in range(4):
        print(f"forked branches, replay {i}", flush=True)
        g.replay()
        cuda.cuda.synchronize()
        p[0].check()
        p[1].check()
        cuda.cuda.synchronize()


def test_two_graphs_of_one_stream_and_eager_calls(cuda, work):
    p, s = work
    g = [capture(cuda, s[0], lambda q=q: q.run(s[0])) for q in p[:2]]
    for i in range(4):
        print(f"two graphs and eager calls, replay {i}", flush=True)
        with cuda.cuda.stream(s[1]):
            g[0].replay()
        g[1].replay()
        p[2].run(s[0])
        cuda.cuda.synchronize()
        for q in p:
            q.check()
        cuda.cuda.synchronize()
