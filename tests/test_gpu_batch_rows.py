"""The batched per-row kernels at the edges of their tiles and runs.

Attention of whole chunks: windows around the 16-key tiles up to the 80-row limit, one key, fresh
streams.  Tolerance: f32 products and sums in another order than the oracle's, 1e-5 of the largest.

Depthwise conv + LN + SiLU of table rows: from 1200 rows on a workgroup takes two table rows, from 3000
on seven, with shared input rows where they lie on consecutive cache rows, so every row has to come out
with the same bits however the table is cut into chunks, ordered or started; the references are the
same row in a table whose neighbours are elsewhere and in tables of one row per workgroup.
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
    dO, dOs, dOff = gpu.alloc(m * D * 4), gpu.alloc(m * D * 4), gpu.alloc(m * D * 4 + 8)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(dh)))
    gpu.begin()
    gpu.check(L.nk_attention_rel_chunks(gpu.h, dkv.ptr, 3 * D, dch.ptr, len(spec), dP.ptr, dbu.ptr, dbv.ptr, dO.ptr, Lmax, H,
                                        dh, D, scale))
    gpu.check(L.nk_attention_rel_chunks_split(gpu.h, dkv.ptr, 3 * D, dch.ptr, len(spec), dP.ptr, dbu.ptr, dbv.ptr, dOs.ptr,
                                              Lmax, H, dh, D, scale))
    gpu.check(L.nk_attention_rel_chunks_split(gpu.h, dkv.ptr, 3 * D, dch.ptr, len(spec), dP.ptr, dbu.ptr, dbv.ptr, dOff.at(2),
                                              Lmax, H, dh, D, scale))  # rows off 8 bytes
    gpu.end()
    out = dO.read((m, D))
    assert rel_err(out, np.concatenate(refs)) < 1e-5
    assert np.array_equal(dOs.read((m, 2 * D), np.uint16), split_rows(out))
    assert np.array_equal(dOff.read((m, 2 * D), np.uint16, 2), split_rows(out))


@pytest.mark.parametrize("rows", [1203, 3002])
@pytest.mark.parametrize("D", [4, 256, 1020, 1024])
@pytest.mark.parametrize("order", ["chunks", "shuffled", "middle", "descending", "gaps"])
def test_dwconv_runs(gpu, D, order, rows):
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
    table = (table * (rows // len(table) + 1))[:rows]
    M = len(table)
    din = rng.standard_normal((pos + 8, D)).astype(np.float32)
    W = (rng.standard_normal((D, 9)) / 3).astype(np.float32)
    g, b = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32), (0.1 * rng.standard_normal(D)).astype(np.float32)
    perm = rng.permutation(M)
    alone = [(table[i][0], 0, 1, 0) for i in perm]
    ddin, dW, dg, db = (gpu.put(x) for x in (din, W, g, b))
    drows, dalone = gpu.put(np.asarray(table, np.int32)), gpu.put(np.asarray(alone, np.int32))
    dY, dYs, dA, dO = (gpu.alloc(M * D * 4) for _ in range(4))
    gpu.begin()
    for m in range(0, M, 1100):  # one row per workgroup
        gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, drows.at(16 * m), min(1100, M - m), dW.ptr, dg.ptr, db.ptr,
                                           dO.at(4 * D * m), D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, drows.ptr, M, dW.ptr, dg.ptr, db.ptr, dY.ptr, D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, dalone.ptr, M, dW.ptr, dg.ptr, db.ptr, dA.ptr, D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows_split(gpu.h, ddin.ptr, drows.ptr, M, dW.ptr, dg.ptr, db.ptr, None, dYs.ptr, D, 9, 1e-5))
    gpu.end()
    y = dY.read((M, D))
    assert np.array_equal(bits(y[perm]), bits(dA.read((M, D))))
    assert np.array_equal(bits(y), bits(dO.read((M, D))))
    assert np.array_equal(dYs.read((M, 2 * D), np.uint16), split_rows(y))
    pick = list(range(90)) + [M - 1]
    ref = np.concatenate([oracle.dwconv_ln_silu(din[table[i][0] - 8:table[i][0] + 1], W, g, b, 1) for i in pick])
    assert rel_err(y[pick], ref) < 1e-5


@pytest.mark.parametrize("M", [5, 1199, 1200, 3001])
def test_dwconv_rows_without_table(gpu, M):
    """No row table: the rows of one run from din_base on, as nk_dwconv_ln_silu, at every row count."""
    import nemoasr

    L = nemoasr.lib()
    D = 64
    rng = np.random.default_rng(M)
    din, W = rng.standard_normal((M + 8, D)).astype(np.float32), (rng.standard_normal((D, 9)) / 3).astype(np.float32)
    g, b = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32), (0.1 * rng.standard_normal(D)).astype(np.float32)
    ddin, dW, dg, db = (gpu.put(x) for x in (din, W, g, b))
    dY, dZ = gpu.alloc(M * D * 4), gpu.alloc(M * D * 4)
    gpu.begin()
    gpu.check(L.nk_dwconv_ln_silu(gpu.h, ddin.ptr, dW.ptr, dg.ptr, db.ptr, dY.ptr, M, D, 9, 1e-5))
    gpu.check(L.nk_dwconv_ln_silu_rows(gpu.h, ddin.ptr, None, M, dW.ptr, dg.ptr, db.ptr, dZ.ptr, D, 9, 1e-5))
    gpu.end()
    assert np.array_equal(bits(dZ.read((M, D))), bits(dY.read((M, D))))


@pytest.mark.parametrize("T,F,C,batch", [(19, 33, 256, 9), (20, 30, 256, 7), (37, 65, 32, 5), (33, 31, 1024, 2), (64, 9, 4, 40)])
def test_dwconv2d_forms(gpu, T, F, C, batch):
    """The four-channel form against the one-channel form (taken for rows off 16 bytes), bit for bit, on
    even and odd sizes, a last group of fewer than four outputs and several segments per workgroup."""
    import nemoasr

    L = nemoasr.lib()
    rng = np.random.default_rng([T, F, C])
    T1, F1 = T // 2 + 1, F // 2 + 1
    assert T1 * F1 * batch >= 256
    X = rng.standard_normal((batch, T, F, C)).astype(np.float32)
    W, b = (rng.standard_normal((C, 9)) / 3).astype(np.float32), rng.standard_normal(C).astype(np.float32)
    dX, dW, db = gpu.put(X), gpu.put(W), gpu.put(b)
    off = gpu.alloc(X.nbytes + 4)
    off.write(X, 4)
    dY, dZ = (gpu.alloc(batch * T1 * F1 * C * 4) for _ in range(2))
    gpu.begin()
    gpu.check(L.nk_dwconv2d_s2_b(gpu.h, dX.ptr, dW.ptr, db.ptr, dY.ptr, T, F, T1, F1, C, batch))
    gpu.check(L.nk_dwconv2d_s2_b(gpu.h, off.at(4), dW.ptr, db.ptr, dZ.ptr, T, F, T1, F1, C, batch))
    gpu.end()
    y = dY.read((batch, T1, F1, C))
    assert np.array_equal(bits(y), bits(dZ.read(y.shape)))
    assert rel_err(y[-1], oracle.dwconv2d_s2(X[-1], W, b)) < 1e-6


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("nwin,batch", [(9, 1), (23, 3), (61, 2), (64, 40)])
def test_convs_skip_taps_outside(gpu, nwin, batch, bad):
    """A tap outside the input is skipped, not multiplied by zero: weights that are infinite or NaN leave
    the outputs that skip them alone.  Every form against the oracle, which skips: the same values
    are infinite and NaN, the rest within 1e-6 (sums of nine products in one order)."""
    import nemoasr

    L = nemoasr.lib()
    F, C = 40, 64
    rng = np.random.default_rng(nwin)
    X = rng.standard_normal((batch, nwin, F)).astype(np.float32)
    W0, W2 = ((rng.standard_normal((C, 9)) / 3).astype(np.float32) for _ in range(2))
    b0, b2 = ((0.1 * rng.standard_normal(C)).astype(np.float32) for _ in range(2))
    for k in range(9):
        W0[k, k] = W2[10 + k, k] = bad
        W0[20 + k, k], W2[20 + k, 8 - k] = bad, bad
    T1, F1 = nwin // 2 + 1, F // 2 + 1
    T2, F2 = T1 // 2 + 1, F1 // 2 + 1
    with np.errstate(all="ignore"):
        y0 = np.stack([oracle.conv2d_c1_s2_relu(x, W0, b0) for x in X])
        ref = np.stack([oracle.dwconv2d_s2(y, W2, b2) for y in y0])
    dX, dW0, db0, dW2, db2, d0 = (gpu.put(x) for x in (X, W0, b0, W2, b2, y0))
    dY, dZ = gpu.alloc(ref.nbytes), gpu.alloc(ref.nbytes)
    gpu.begin()
    gpu.check(L.nk_conv2d_c1_dw_s2_b(gpu.h, dX.ptr, dW0.ptr, db0.ptr, dW2.ptr, db2.ptr, dY.ptr, nwin, F, T1, F1, T2, F2, C, batch))
    gpu.check(L.nk_dwconv2d_s2_b(gpu.h, d0.ptr, dW2.ptr, db2.ptr, dZ.ptr, T1, F1, T2, F2, C, batch))
    gpu.end()
    for got in (dY.read(ref.shape), dZ.read(ref.shape)):
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)]) and np.array_equal(np.isinf(got), np.isinf(ref))
        assert rel_err(got[np.isfinite(ref)], ref[np.isfinite(ref)]) < 1e-6


@pytest.mark.parametrize("T,F,C,batch", [(10, 17, 256, 12), (3, 5, 1016, 33), (9, 11, 36, 141)])
def test_flatten_forms(gpu, T, F, C, batch):
    """Through LDS (half a million elements or more) and element by element: the transpose itself."""
    import nemoasr

    L = nemoasr.lib()
    assert T * F * C * batch >= 500000
    X = np.random.default_rng(T).standard_normal((batch, T, F, C)).astype(np.float32)
    dX, dY, dZ = gpu.put(X), gpu.alloc(X.nbytes), gpu.alloc(X[0].nbytes)
    gpu.begin()
    gpu.check(L.nk_flatten_cf_b(gpu.h, dX.ptr, dY.ptr, T, F, C, batch))
    gpu.check(L.nk_flatten_cf_b(gpu.h, dX.ptr, dZ.ptr, T, F, C, 1))
    gpu.end()
    ref = np.ascontiguousarray(X.transpose(0, 1, 3, 2)).reshape(batch, T, C * F)
    assert np.array_equal(dY.read(ref.shape), ref)
    assert np.array_equal(dZ.read(ref[0].shape), ref[0])
