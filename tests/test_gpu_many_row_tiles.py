"""Every tile of the many-row GEMM against the 64x64 one, bit for bit, and against float64.

The tiles differ in their wavefront layout, ring depth and in whether separate wavefronts load, but
sum K in the same order, so a row's result must not depend on the tile the host picks for the row
count.  Sizes: rows around the tile edges, the shortest K loops (one step, fewer steps than ring
stages, a last step of 32 columns with f32 rows), more workgroups than one round holds.
Tolerance against float64: activations carry 16 significant bits (2^-17 relative rounding) and the
K sums are f32, so 2e-5 of the largest result.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_err
from test_gpu_split import bits, split_rows, w_bf16

pytestmark = pytest.mark.gpu

TILES = [0, 1, 2, 3, 4, 5, 6, 7, 8, -1]


def reference(A, W, bias, act, split):
    A = A.astype(np.float64)
    if split:
        hi = oracle.bf16_to_f32(oracle.f32_to_bf16(A.astype(np.float32))).astype(np.float64)
        A = hi + oracle.bf16_to_f32(oracle.f32_to_bf16((A - hi).astype(np.float32)))
    y = A @ oracle.bf16_to_f32(W).astype(np.float64).T
    if bias is not None:
        y = y + bias
    if act == 1:
        y = y / (1 + np.exp(-y))
    elif act == 2:
        y = np.maximum(y, 0)
    elif act == 3:
        n = y.shape[1] // 2
        y = y[:, :n] / (1 + np.exp(-y[:, n:]))
    return y


@pytest.mark.parametrize("M,N,K", [(17, 256, 64), (32, 256, 128), (33, 512, 704), (64, 256, 1024), (65, 1024, 192),
                                   (97, 512, 320), (129, 512, 1024), (300, 2048, 256), (18, 256, 96), (65, 256, 32), (70, 512, 1056),
                                   (50, 256, 2048)])
@pytest.mark.parametrize("form", ["plain", "bias_relu", "silu_split", "glu_rows", "odd_ldc", "resid", "resid_unsplit"])
def test_tiles_agree(gpu, M, N, K, form):
    """resid_unsplit: the K blocks one after another on every tile (partial rows read back)."""
    import nemoasr

    L = nemoasr.lib()
    ksplit = 0 if form == "resid_unsplit" else -1
    form = form.removesuffix("_unsplit")
    rng = np.random.default_rng([M, N, K])
    A = rng.standard_normal((M, K)).astype(np.float32)
    W = w_bf16(rng, N, K)
    bias = (0.1 * rng.standard_normal(N)).astype(np.float32) if form == "bias_relu" else None
    act = {"bias_relu": 2, "silu_split": 1, "glu_rows": 3}.get(form, 0)
    nout = N // 2 if act == 3 else N
    crow = rng.permutation(M + 5)[:M].astype(np.int32) if form == "glu_rows" else None
    rows, ldc = (M + 5 if crow is not None else M), nout + (1 if form == "odd_ldc" else 0)
    C0 = rng.standard_normal((rows, ldc)).astype(np.float32)
    dW, dB = gpu.put(W), gpu.put(bias) if bias is not None else None
    dR = gpu.put(crow) if crow is not None else None
    for split in (False, True):
        if split and K % 64:
            continue
        dA = gpu.put(split_rows(A) if split else A)
        got = {}
        for tile in TILES:
            dC = gpu.alloc(M * 4 * nout) if form == "silu_split" else gpu.put(C0)
            prev, prev_split = L.nk_gemm_mx_tile(tile), L.nk_gemm_ksplit(ksplit)
            try:
                gpu.begin()
                gpu.check(L.nk_gemm_split(
                    gpu.h, None if split else dA.ptr, dA.ptr if split else None, 2 * K if split else K, dW.ptr, K,
                    dB.ptr if dB else None, None if form == "silu_split" else dC.ptr,
                    dC.ptr if form == "silu_split" else None, 2 * nout if form == "silu_split" else ldc,
                    dR.ptr if dR else None, M, N, K, act, int(form == "resid"), 0.5 if form == "resid" else 1.0))
                gpu.end()
            finally:
                L.nk_gemm_mx_tile(prev)
                L.nk_gemm_ksplit(prev_split)
            got[tile] = dC.read((M, 2 * nout), np.uint16) if form == "silu_split" else dC.read((rows, ldc))
            dC.free()
        for tile in TILES:
            assert np.array_equal(bits(got[tile]), bits(got[2])), (split, tile)
        ref = reference(A, W, bias, act, split)
        if form == "silu_split":
            v = oracle.bf16_to_f32(got[2][:, :nout]).astype(np.float64) + oracle.bf16_to_f32(got[2][:, nout:])
        else:
            v = got[2][crow] if crow is not None else got[2][:, :nout]
            if form == "resid":
                ref = C0 + 0.5 * ref
        assert rel_err(v, ref) < 2e-5, split
        if crow is not None:  # rows outside the map stay
            rest = np.setdiff1d(np.arange(rows), crow)
            assert np.array_equal(got[2][rest], C0[rest])
        if form == "odd_ldc":
            assert np.array_equal(got[2][:, nout], C0[:, nout])
        dA.free()


@pytest.mark.parametrize("form", ["plain", "glu", "resid"])
def test_more_tiles_than_the_reciprocals_cover(gpu, form):
    """65536 workgroups and more: the kernels divide instead of multiplying by reciprocals (exact below
    that).  16421 rows on 32x32 (GLU: 32x64) tiles against 64x64, all of them, bit for bit."""
    import nemoasr

    L = nemoasr.lib()
    M, N, K = 16421, 4096, 64
    if form == "glu":
        M *= 2
    if form == "resid":
        M, N, K = 16421, 2048, 1024  # two K blocks
    rng = np.random.default_rng(len(form))
    nout = N // 2 if form == "glu" else N
    dA = gpu.put(split_rows(rng.standard_normal((M, K)).astype(np.float32)))
    dW = gpu.put(w_bf16(rng, N, K))
    tile, tiles = (3, -(-M // 32) * (nout // 32)) if form == "glu" else (4, -(-M // 32) * (nout // 32))
    assert tiles * (2 if form == "resid" else 1) >= 65536
    got = []
    prev_split = L.nk_gemm_ksplit(1 if form == "resid" else -1)
    try:
        for t in (tile, 2):
            dC = gpu.alloc(M * nout * 4)
            gpu.begin()
            gpu.check(L.nk_fill(gpu.h, dC.ptr, M * nout, 0.5))
            prev = L.nk_gemm_mx_tile(t)
            try:
                gpu.check(L.nk_gemm_split(gpu.h, None, dA.ptr, 2 * K, dW.ptr, K, None, dC.ptr, None, nout, None, M, N, K,
                                          3 if form == "glu" else 0, int(form == "resid"), 1.0))
            finally:
                L.nk_gemm_mx_tile(prev)
            gpu.end()
            got.append(dC.read((M, nout)))
            dC.free()
    finally:
        L.nk_gemm_ksplit(prev_split)
        dA.free()
        dW.free()
    assert np.array_equal(bits(got[0]), bits(got[1]))
