"""The batched per-row kernels at the edges of their tiles.

Attention of whole chunks: windows around the 16-key tiles up to the 80-row limit, one key, fresh
streams.  Tolerance: f32 products and sums in another order than the oracle's, 1e-5 of the largest.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_err
from test_gpu_split import split_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [[(1, 0), (2, 0), (16, 0), (16, 64), (1, 79)], [(5, 11), (6, 11), (8, 56), (9, 56), (7, 25)],
                                  [(16, 1), (15, 17), (13, 35), (12, 68), (4, 60)]])
def test_attention_chunk_edges(gpu, spec):
    import nemoasr

    L = nemoasr.lib()
    H, dh, D, Lmax, cap = 2, 128, 256, 82, 96
    rng = np.random.default_rng(len(spec) + spec[0][0])
    kv = rng.standard_normal((len(spec) * cap, 3 * D)).astype(np.float32)
    P = rng.standard_normal((2 * Lmax - 1, D)).astype(np.float32)
    bu, bv = ((0.1 * rng.standard_normal(D)).astype(np.float32) for _ in range(2))
    chunks, refs, m = [], [], 0
    for s, (c, cached) in enumerate(spec):
        pos = s * cap + cached
        K, V = kv[pos - cached:pos + c, D:2 * D], kv[pos - cached:pos + c, 2 * D:]
        refs.append(oracle.attention_rel(kv[pos:pos + c, :D], K, V, P, bu, bv, c, cached + c, Lmax, H, dh))
        chunks += [pos, m, c, cached]
        m += c
    dkv, dP, dbu, dbv, dch = (gpu.put(x) for x in (kv, P, bu, bv, np.asarray(chunks, np.int32)))
    dO, dOs = gpu.alloc(m * D * 4), gpu.alloc(m * D * 4)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(dh)))
    gpu.begin()
    gpu.check(L.nk_attention_rel_chunks(gpu.h, dkv.ptr, 3 * D, dch.ptr, len(spec), dP.ptr, dbu.ptr, dbv.ptr, dO.ptr, Lmax, H,
                                        dh, D, scale))
    gpu.check(L.nk_attention_rel_chunks_split(gpu.h, dkv.ptr, 3 * D, dch.ptr, len(spec), dP.ptr, dbu.ptr, dbv.ptr, dOs.ptr,
                                              Lmax, H, dh, D, scale))
    gpu.end()
    out = dO.read((m, D))
    assert rel_err(out, np.concatenate(refs)) < 1e-5
    assert np.array_equal(dOs.read((m, 2 * D), np.uint16), split_rows(out))
