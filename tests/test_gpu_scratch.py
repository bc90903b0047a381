"""The context's split-K scratch: graphs captured before it grows, and launches it is too small for.

A captured residual update holds the address of the scratch its partial rows go to.  A later, larger
update grows the scratch; the graph must then still write memory that belongs to the context.  Where the scratch cannot grow (a capture, the fixed region of the
allocation-free entry point) the K blocks run one after another, on a tile picked for that.
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


def count(L, g, kernel, launch):
    """Launches of a kernel (a name, or a prefix ending in *) during launch()."""
    import ctypes as C

    ms, n, by = C.c_double(), C.c_int(), C.c_double()
    assert L.gpu_timing_set(g.h, kernel.encode(), 16) == 0
    try:
        launch()
        assert L.gpu_timing_collect(g.h, C.byref(ms), C.byref(n), C.byref(by)) == 0
    finally:
        L.gpu_timing_set(g.h, None, 0)
    return n.value


@pytest.mark.parametrize("M,form", [(1536, "noalloc"), (1537, "noalloc"), (600, "capture"), (1000, "capture")])
def test_unsplit_where_the_scratch_is_too_small(clean_gpu, M, form):
    """The tile of split K blocks is not the one for blocks one after another: the pick is made again, and
    the bits are those of the split."""
    import nemoasr

    g, L = clean_gpu, nemoasr.lib()
    rng = np.random.default_rng(M)
    A, C0 = split_rows(rng.standard_normal((M, K)).astype(np.float32)), rng.standard_normal((M, N)).astype(np.float32)
    dW, dA, dC = g.put(w_bf16(rng, N, K)), g.put(A), g.put(C0)
    def noalloc():
        g.begin()
        g.check(L.nk_gemm_split_noalloc(g.h, None, dA.ptr, 2 * K, dW.ptr, K, None, dC.ptr, None, N, None, M, N, K, 0, 1, 0.5))
        g.end()

    if form == "noalloc":
        assert count(L, g, "gemm_mx64x128*", noalloc) == 1  # the split's tile: 96x256
        outs = [dC.read((M, N))]
    else:
        g.begin()
        g.check(L.gpu_capture_begin(g.h))
        resid(L, g, dA, dW, dC, M)
        graph = L.gpu_capture_end(g.h)
        g.end()
        assert graph
        outs = []
        for _ in range(3):
            dC.write(C0)
            g.begin()
            g.check(L.gpu_graph_launch(g.h, graph))
            g.end()
            outs.append(dC.read((M, N)))
        L.gpu_graph_free(graph)
    prev = L.nk_gemm_ksplit(1)
    try:
        dC.write(C0)
        g.begin()
        resid(L, g, dA, dW, dC, M)
        g.end()
    finally:
        L.nk_gemm_ksplit(prev)
    ref = dC.read((M, N))
    for y in outs:
        assert np.array_equal(bits(y), bits(ref))


@pytest.fixture
def clean_gpu():
    import nemoasr

    g = nemoasr.Gpu()
    yield g
    g.close()
