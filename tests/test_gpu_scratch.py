"""The context's split-K scratch: graphs captured before it grows.

A captured residual update holds the address of the scratch its partial rows go to.  A later, larger
update grows the scratch; the graph must then still write memory that belongs to the context.
"""
import numpy as np
import pytest

from test_gpu_split import bits, split_rows, w_bf16

pytestmark = pytest.mark.gpu

N, K = 1024, 4096


def resid(L, g, dA, dW, dC, M):
    g.check(L.nk_gemm_split(g.h, None, dA.ptr, 2 * K, dW.ptr, K, None, dC.ptr, None, N, None, M, N, K, 0, 1, 0.5))


def test_graph_outlives_scratch_growth(clean_gpu):
    import nemoasr

    g, L = clean_gpu, nemoasr.lib()
    rng = np.random.default_rng(5)
    dW = g.put(w_bf16(rng, N, K))
    graphs = []
    prev = L.nk_gemm_ksplit(1)  # four parts: 100 rows fit the scratch of a new context, 300 and 700 do not
    try:
        for M in (100, 300, 700):
            C0 = rng.standard_normal((M, N)).astype(np.float32)
            dA, dC = g.put(split_rows(rng.standard_normal((M, K)).astype(np.float32))), g.put(C0)
            g.begin()
            resid(L, g, dA, dW, dC, M)  # grows the scratch, which the graphs before it do not know
            g.end()
            ref = dC.read((M, N))
            g.begin()
            g.check(L.gpu_capture_begin(g.h))
            resid(L, g, dA, dW, dC, M)
            graph = L.gpu_capture_end(g.h)
            g.end()
            assert graph
            graphs.append((M, C0, dC, ref, graph))
        # memory a freed block would have gone to
        mark = np.full(1 << 20, -7.25, np.float32)
        others = [g.put(mark) for _ in range(16)]
        for _ in range(3):
            for M, C0, dC, ref, graph in graphs:
                dC.write(C0)
                g.begin()
                g.check(L.gpu_graph_launch(g.h, graph))
                g.end()
                assert np.array_equal(bits(dC.read((M, N))), bits(ref)), M
            for o in others:
                assert np.array_equal(o.read(mark.shape), mark)
    finally:
        L.nk_gemm_ksplit(prev)
        for *_, graph in graphs:
            L.gpu_graph_free(graph)


@pytest.fixture
def clean_gpu():
    import nemoasr

    g = nemoasr.Gpu()
    yield g
    g.close()
