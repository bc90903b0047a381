"""The batched per-row kernels at the edges of their tiles and runs.

Attention of whole chunks: windows around the 16-key tiles up to the 80-row limit, one key, fresh
streams.  Tolerance: f32 products and sums in another order than the oracle's, 1e-5 of the largest.

Depthwise conv + LN + SiLU of table rows: from 1200 rows on a workgroup takes seven table rows, with
shared input rows where they lie on consecutive cache rows, so every row has to come out with the same
bits however the table is cut into chunks, ordered or started; the reference is the same row in a
table whose neighbours are elsewhere.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_err
from test_gpu_split import bits, split_rows

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


@pytest.mark.parametrize("D", [4, 256, 1020, 1024])
@pytest.mark.parametrize("order", ["chunks", "shuffled", "middle", "descending", "gaps"])
def test_dwconv_runs(gpu, D, order):
    import nemoasr

    L = nemoasr.lib()
    rng = np.random.default_rng([D, len(order)])
    table, pos = [], 8
    for c in [7, 1, 14, 2, 8, 13, 4, 16, 6, 15]:
        table += [(pos + i, i, c, 56) for i in range(c)]
        pos += c + 8
    if order == "shuffled":
        table = [table[i] for i in rng.permutation(len(table))]
    elif order == "middle":
        table = table[3:6] + table[9:20] + table[25:]
    elif order == "descending":
        table = table[::-1]
    elif order == "gaps":  # indices that go on while the cache rows do not, and the reverse
        table = [(r + (i > 2), i + (i > 4), c, k) for r, i, c, k in table]
    table = (table * (1200 // len(table) + 1))[:1203]
    M = len(table)
    din = rng.standard_normal((pos + 8, D)).astype(np.float32)
    W = (rng.standard_normal((D, 9)) / 3).astype(np.float32)
    g, b = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32), (0.1 * rng.standard_normal(D)).astype(np.float32)
    perm = rng.permutation(M)
    alone = [(table[i][0], 0, 1, 0) for i in perm]
    ddin, dW, dg, db = (gpu.put(x) for x in (din, W, g, b))
    drows, dalone = gpu.put(np.asarray(table, np.int32)), gpu.put(np.asarray(alone, np.int32))
    dY, dYs, dA = (gpu.alloc(M * D * 4) for _ in range(3))
    gpu.begin()
    gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, drows.ptr, M, dW.ptr, dg.ptr, db.ptr, dY.ptr, D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, dalone.ptr, M, dW.ptr, dg.ptr, db.ptr, dA.ptr, D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows_split(gpu.h, ddin.ptr, drows.ptr, M, dW.ptr, dg.ptr, db.ptr, None, dYs.ptr, D, 9, 1e-5))
    gpu.end()
    y = dY.read((M, D))
    assert np.array_equal(bits(y[perm]), bits(dA.read((M, D))))
    assert np.array_equal(dYs.read((M, 2 * D), np.uint16), split_rows(y))
    pick = list(range(90)) + [M - 1]
    ref = np.concatenate([oracle.dwconv_ln_silu(din[table[i][0] - 8:table[i][0] + 1], W, g, b, 1) for i in pick])
    assert rel_err(y[pick], ref) < 1e-5
