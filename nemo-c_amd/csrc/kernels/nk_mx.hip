/* Many-row bf16-weight GEMM for gfx950, fed by direct global -> LDS loads (M > 16: the batched
 * multi-stream encoder and decoder): C[crow(m)][n] (= or +=) alpha * act(A W^T + b); GLU pairs
 * weight rows n and n + N/2.
 *
 * Workgroup tile BM x BN computed by WGM (along M) x WGN (along N) wavefronts; each owns a
 * (BM/WGM) x (BN/WGN) block of 16x16 tiles of v_mfma_f32_16x16x32_bf16.
 *
 * Operand staging: a ring of NS LDS stages, each holding one K step of 64 columns of A (two planes
 * of BM x 128 B) and W (BN x 128 B).  Stages are filled by global_load_lds_dwordx4 (16 bytes per lane
 * straight into LDS, no registers), up to NS-1 steps ahead of their use.  A DMA instruction writes 64
 * consecutive 16-byte LDS granules in lane order; the global address each lane reads is chosen so
 * that granule g of row r holds K-granule (g ^ swizzle(r)), which makes the 16-row fragment reads
 * (ds_read_b128) hit distinct banks (swz_a / swz_h below).
 *
 * What bounds it, and the two forms (PW).  With one 4-wavefront workgroup on a CU a step of a 64x64
 * tile took 0.38 us (wall clock stamps per step) where its MFMAs take 0.1 us and its LDS traffic
 * 0.24 us: a wavefront that issues its share of the loads is stalled 70-120 cycles per DMA
 * instruction (four wavefronts on a CU stream 138 GB/s, eight 217, sixteen 323, measured from L2)
 * and then waits for its fragment reads.
 *   - PW = 4: four more wavefronts only load, so the computing ones never issue a DMA; 18 rows,
 *     FF up 10.6 -> 6.6 us, 448 rows, FF up 15.9 -> 13.8, FF down 13.8 -> 12.1.  All tiles but three.
 *   - PW = 0: 128x256 and 96x256 computed and loaded by eight wavefronts (two per SIMD, 198 VGPRs
 *     each: no room for loaders; 192x256 spills), half the staged bytes per MFMA of 64x128: the steps of
 *     128x256 take 1.7 us, 1.26 PFLOP/s issued (a large library product here: 1.13); 3584 rows, FF up
 *     81.7 -> 69 us, pw1 40.4 -> 29.2 us.  64x128u by four, which keep two sets of sums.
 * In both, a step's fragments are in registers one 32-K substep ahead of their MFMAs, so LDS latency
 * is covered by the other substep's MFMAs; the accumulators stay in VGPRs; the weights are the
 * MFMA's first operand, so a lane holds four consecutive output columns and stores 8 or 16 bytes at
 * once.  What is left at few rows is fixed: ~0.6 us of start (arguments, instruction fetch) before
 * the first load, ~1.7 us between graph nodes; at many rows the tile count against 256 CUs.
 *
 * A enters the MFMAs as bf16 hi = RNE(a) and lo = RNE(a - hi), and every K step issues the hi and
 * the lo product: 16 significant bits of A against exact bf16 weights, f32 accumulation.  The
 * reference's many-row path multiplies f32 A by bf16 W in f32 (src/kernels.metal:120-208,
 * simdgroup_float8x8).  Two A forms:
 *   - f32 rows (AS = false): each fragment (8 consecutive K of one row per lane) is split in
 *     registers (v_cvt_pk_bf16_f32) after its LDS read;
 *   - split rows (AS = true, NkGemmArgs.A2): the producer stored hi and lo (the same values), so
 *     both planes stream into LDS like the weights and the fragments feed the MFMAs directly, with
 *     no VALU work in the K loop.
 * A kernel that produces the next GEMM's A can write split rows itself (OS, NkGemmArgs.C2).
 *
 * Tile order: the grid is 8 x (tiles per XCD); workgroup b runs on XCD b % 8 and takes tile
 * (b % 8) * per + b / 8 of an order that walks groups of group_m row tiles across all column tiles
 * (row tile fastest), so the workgroups of one XCD share weight columns and a few row panels in
 * that XCD's L2.  grid tiles past the end exit at once.
 *
 * Accumulating GEMMs without bias or activation (the residual updates: C += alpha * A W^T) run on
 * the _acc kernels.  They sum K in kblocks equal blocks, each from zero, and add the block sums in
 * block order; with splits = kblocks every workgroup computes one block.  Either way the kernel
 * only writes partial rows (one per split), and the update C + alpha * (((0 + p0) + p1) + ...) is
 * applied by the next kernel that reads C (the batched encoder's LayerNorms) or by resid_fold.
 * Both forms give the same bits, so the host may split K or not by the row count (how many other
 * streams share the step) without changing any row's result, and no result depends on which
 * workgroup finishes first; no workgroup waits for or communicates with another. */
#include "nk_common.h"

/* LDS granule swizzles: granule g of row r lives in slot g ^ swz(r).  A fragment read is one
 * ds_read_b128 per lane over 16 consecutive rows at one K granule (lanes 16 f .. 16 f + 15).  f32
 * rows of 8 granules (32 K): chosen by the SQ_LDS_BANK_CONFLICT counter on gfx950 over candidate
 * functions; it reads with zero conflict cycles, where ((r>>1)&7)^((r&1)<<2) costs 4 extra cycles
 * per read (a 2-way conflict; 1-3% of kernel time) and the plain r % 8 cost a third of the kernel
 * time at 3584 rows. */
__device__ __forceinline__ u32 swz_a(u32 r) { return (r & 7) ^ ((r >> 3) & 1); }
/* bf16 rows of 8 granules (64 K): the f32 rows' geometry but another read pattern (lane group f reads
 * granule 4h + f, not 2f and 2f + 1): swz_a costs a 2-way conflict on every read there, (r >> 1) & 7
 * none */
__device__ __forceinline__ u32 swz_h(u32 r) { return (r >> 1) & 7; }
/* waits until at most rem <= R steps of L loads each are in flight */
template <int R, int L> __device__ __forceinline__ void wait_steps(u32 rem) {
    if constexpr (R > 0)
        if (rem < (u32)R) {
            wait_steps<R - 1, L>(rem);
            return;
        }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R * L) : "memory");
}
/* x / d by the reciprocal of d the host computed (NkGemmArgs.rc_*) */
__device__ __forceinline__ u32 div_rc(u32 x, u32 rc) { return rc ? __umulhi(x, rc) : x; }
__device__ __forceinline__ void wait_lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

/* PW: wavefronts that only load (0: the computing ones load).
 * EPI: 0 bias / activation / GLU / accumulate epilogue; 1 argmax keys; 2 blocked-K residual
 * update into partial rows (TOT: the sum of several blocks stays in registers).  AS: A as split rows; OS: outputs as split rows (EPI 0 without GLU). */
template <int BM, int BN, int WGM, int WGN, int PW, int NS, bool GLU, int EPI, bool AS, bool OS, bool TOT = false>
__device__ __forceinline__ void mx_impl(const NkGemmArgs &a, lds_char_t *const smem) {
    static_assert(!OS || (EPI == 0 && !GLU), "split outputs from the plain epilogue only");
    constexpr int NW = PW ? PW : WGM * WGN, KS = NK_MX_KS; /* NW: wavefronts that load */
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int TI = WTM / 16, TJ = WTN / 16;
    constexpr u32 PLANE = BM * 128;          /* one plane of A: BM rows of 128 bytes */
    constexpr u32 STAGE = 2 * PLANE + BN * 128;
    constexpr int AI = BM / 4 / NW;          /* DMA instructions per wavefront per stage: A, W */
    constexpr int BI = BN / 8 / NW;
    static_assert(AI >= 1 && BI >= 1 && TI >= 1 && TJ >= (GLU ? 2 : 1), "tile shape");
    static_assert(AI * NW * 4 == BM && BI * NW * 8 == BN && TI * 16 * WGM == BM && TJ * 16 * WGN == BN, "tile shape");
    static_assert(EPI != 2 || !GLU, "the residual update has no GLU");
    static_assert((NS - 1) * (AI + BI) < 64, "vmcnt range");
    const u32 tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = PW && wv >= WGM * WGN;
    const u32 wave = loader ? wv - WGM * WGN : wv;
    const u32 wm = wave / WGN, wn = wave % WGN;
    const u32 M = a.mrows ? min(a.M, (u32)max(*a.mrows, 0) * a.mrows_mul) : a.M;
    const u32 nout = GLU ? a.N / 2 : a.N, KZ = a.splits;

    /* tile of this workgroup */
    const u32 per = gridDim.x / 8;
    const u32 t = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const u32 TMt = EPI != 1 && a.tm ? a.tm : (M + BM - 1) / BM, TNt = nout / (GLU ? BN / 2 : BN);
    if (t >= TMt * TNt * KZ) return;
    const u32 G = a.group_m, gsz = G * TNt;
    u32 kz, tt, grp, within, gh, tn;
    if (EPI != 1 && a.tm) {
        kz = div_rc(t, a.rc_mn), tt = t - kz * TMt * TNt;
        grp = div_rc(tt, a.rc_grp), within = tt - grp * gsz;
        gh = min(TMt - grp * G, G);
        tn = div_rc(within, gh == G ? a.rc_gm : a.rc_last);
    } else {
        kz = t / (TMt * TNt), tt = t % (TMt * TNt);
        grp = tt / gsz, within = tt % gsz;
        gh = min(TMt - grp * G, G);
        tn = within / gh;
    }
    const u32 tm = grp * G + within - tn * gh;
    const u32 m0 = tm * BM;
    const u32 c0 = tn * (GLU ? BN / 2 : BN); /* first output column */
    /* K steps; a last step of 32 columns (K % 64 == 32, f32 A only) has one substep */
    const u32 S = (a.K + KS - 1) / KS;
    const bool half = !AS && (a.K & 32);
    const u32 s_begin = (u32)(((u64)S * kz) / KZ), s_end = (u32)(((u64)S * (kz + 1)) / KZ);
    const u32 nst = s_end - s_begin;
    /* K steps per block of the blocked sum (EPI 2; the whole range otherwise) */
    const u32 spb = EPI == 2 ? S / a.kblocks : nst;

    /* DMA sources: granule p of a stage region is written by lane p % 64 of instruction p / 64
     * (instruction j of wavefront w covers p in [(NW j + w) * 64, +64)).  The A region is two planes of
     * BM rows of 8 granules: split A the hi then the lo plane of 64 K, f32 A the first then the second
     * 32 K. */
    const char *asrc[AI], *bsrc[BI];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const u32 p = (NW * j + wave) * 64 + lane, plane = p / (BM * 8), q = p % (BM * 8), r = q / 8;
        if constexpr (AS)
            asrc[j] = (const char *)(a.A2 + (u64)min(m0 + r, M - 1) * a.lda + plane * a.K + 8 * ((q & 7) ^ swz_h(r)) +
                                     (u64)s_begin * KS);
        else
            asrc[j] = (const char *)(a.A + (u64)min(m0 + r, M - 1) * a.lda + plane * 32 + 4 * ((q & 7) ^ swz_a(r)) +
                                     (u64)s_begin * KS);
    }
    constexpr u32 A_STEP = AS ? KS * 2 : KS * 4; /* bytes of one K step of one A row (per plane) */
#pragma unroll
    for (int j = 0; j < BI; ++j) {
        const u32 p = (NW * j + wave) * 64 + lane, n = p / 8, kg = (p & 7) ^ swz_h(n);
        u32 col;
        if (GLU) col = n < BN / 2 ? c0 + n : a.N / 2 + c0 + (n - BN / 2);
        else col = c0 + n;
        bsrc[j] = (const char *)(a.W + (u64)col * a.ldw + 8 * kg + (u64)s_begin * KS);
    }
    /* loads of the next K step (`last`: the final one) into the stage at `st`; the sources advance */
    auto issue = [&](lds_char_t *st, bool last) {
        if (half && last) { /* the second 32 columns do not exist: load the first ones again, unused */
#pragma unroll
            for (int j = 0; j < AI; ++j)
                dma16(asrc[j] - ((NW * j + wave) * 64 + lane >= BM * 8 ? 128 : 0), st + (NW * j + wave) * 1024);
#pragma unroll
            for (int j = 0; j < BI; ++j) {
                const u32 p = (NW * j + wave) * 64 + lane;
                dma16(bsrc[j] - (((p & 7) ^ swz_h(p / 8)) >= 4 ? 64 : 0), st + 2 * PLANE + (NW * j + wave) * 1024);
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < AI; ++j) {
            dma16(asrc[j], st + (NW * j + wave) * 1024);
            asrc[j] += A_STEP;
        }
#pragma unroll
        for (int j = 0; j < BI; ++j) {
            dma16(bsrc[j], st + 2 * PLANE + (NW * j + wave) * 1024);
            bsrc[j] += KS * 2;
        }
    };
    /* fragment addresses inside a stage: row 16 i + lane % 16 of the wavefront's block, K granule
     * lane / 16; the swizzle of rows 16 apart is the same, so the rest are constant offsets */
    const u32 fr = lane & 15, fg = lane >> 4;
    u32 ao[2], bo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const u32 sp = ((4 * h + fg) ^ swz_h(fr)) * 16;
        /* split A: substep h; f32 A: the two halves of a fragment's 8 columns */
        ao[h] = (wm * WTM + fr) * 128 + (AS ? sp : ((2 * fg + h) ^ swz_a(fr)) * 16);
        bo[h] = 2 * PLANE + (wn * (GLU ? WTN / 2 : WTN) + fr) * 128 + sp;
    }
    struct frags { uint4 b[TJ], h[TI], l[TI]; } F[2];
    auto read = [&](frags &f, const lds_char_t *st, int h) { /* substep h of the stage at st */
        typedef const __attribute__((address_space(3))) uint4 *lds4;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const u32 n = GLU ? (j < TJ / 2 ? 16 * j : BN / 2 + 16 * (j - TJ / 2)) : 16 * j;
            f.b[j] = *(lds4)(st + bo[h] + n * 128);
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            if constexpr (AS) {
                f.h[i] = *(lds4)(st + ao[h] + 16 * i * 128);
                f.l[i] = *(lds4)(st + ao[h] + 16 * i * 128 + PLANE);
            } else { /* the f32 values; split when they are used */
                f.h[i] = *(lds4)(st + ao[0] + 16 * i * 128 + h * PLANE);
                f.l[i] = *(lds4)(st + ao[1] + 16 * i * 128 + h * PLANE);
            }
        }
    };

    floatx4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = (floatx4){ 0.f, 0.f, 0.f, 0.f };
    /* lane l holds row 16 i + l % 16, columns 16 j + 4 (l / 16) + e of each tile */
    const u32 row0 = m0 + wm * WTM + fr;
    /* EPI 2, the residual update, deferred: the K blocks' sums go to partials[kz][row][n] (rows of N
     * floats), (((0 + b0) + b1) + ...) where one workgroup computes several.  The rows are folded
     * into C in block order afterwards, by the LayerNorm that reads them next or by resid_fold:
     * C + alpha * (((0 + p0) + p1) + ...), the unsplit epilogue's bits.  The sum so far is kept in
     * registers (TOT: for kernels that run several blocks per workgroup) or read back from the
     * partial row (kernels that run several only where the scratch holds no more parts). */
    floatx4 tot[TOT ? TI : 1][TOT ? TJ : 1];
    if constexpr (TOT)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) tot[i][j] = (floatx4){ 0.f, 0.f, 0.f, 0.f };
    auto end_block = [&](bool first, bool last) {
        float *P = a.ws + (u64)kz * a.M * a.N + c0 + wn * WTN + 4 * fg;
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const bool in = row0 + 16 * i < M;
            floatx4 *p = (floatx4 *)(P + (u64)(in ? row0 + 16 * i : M - 1) * a.N);
            floatx4 t[TJ];
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                if constexpr (TOT) t[j] = tot[i][j];
                else t[j] = first ? (floatx4){ 0.f, 0.f, 0.f, 0.f } : p[4 * j];
            }
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                t[j] += acc[i][j];
                if constexpr (TOT) tot[i][j] = t[j];
                if (in && (!TOT || last)) p[4 * j] = t[j];
                acc[i][j] = (floatx4){ 0.f, 0.f, 0.f, 0.f };
            }
        }
    };
    /* one 32-K substep: every hi product, then every lo product (the same order in every kernel, so
     * every tile gives the same bits).  The weights are the MFMA's first operand: a lane then holds
     * four consecutive output columns of one row */
    auto mma = [&](frags &f) {
        if constexpr (!AS) {
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const float x[8] = { __uint_as_float(f.h[i].x), __uint_as_float(f.h[i].y), __uint_as_float(f.h[i].z),
                                     __uint_as_float(f.h[i].w), __uint_as_float(f.l[i].x), __uint_as_float(f.l[i].y),
                                     __uint_as_float(f.l[i].z), __uint_as_float(f.l[i].w) };
                split8(x, f.h[i], f.l[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j] = mfma_bf16(f.b[j], f.h[i], acc[i][j]);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j] = mfma_bf16(f.b[j], f.l[i], acc[i][j]);
    };

    /* K loop.  A step's second fragments are read while the first multiply, and the next step's first
     * ones while the second multiply; between the two a wavefront waits for its loads of the next
     * step and for its own reads of this one, and the barrier then publishes the next stage and
     * frees this one, which takes the loads of NS steps ahead. */
    if (!PW || loader) {
        for (u32 u = 0; u < min(nst, (u32)NS); ++u) issue(smem + u * STAGE, s_begin + u + 1 == S);
        wait_steps<NS - 1, AI + BI>(min(nst, (u32)NS) - 1);
    }
    barrier_mem();
    if (loader) {
        u32 off = 0;
        for (u32 q = 0; q + 1 < nst; ++q) {
            wait_steps<NS - 2, AI + BI>(min(nst, q + NS) - (q + 2));
            barrier_mem();
            if (q + NS < nst) issue(smem + off, s_begin + q + NS + 1 == S);
            off = off + STAGE == NS * STAGE ? 0 : off + STAGE;
        }
        return;
    }
    read(F[0], smem, 0);
    u32 off = 0;
    for (u32 q = 0; q < nst; ++q) {
        const bool whole = !half || s_begin + q + 1 < S;
        if (whole) read(F[1], smem + off, 1);
        mma(F[0]);
        if (q + 1 < nst) {
            wait_lgkm0();
            if (!PW) wait_steps<NS - 2, AI + BI>(min(nst, q + NS) - (q + 2));
            barrier_mem();
            if (!PW && q + NS < nst) issue(smem + off, s_begin + q + NS + 1 == S);
            off = off + STAGE == NS * STAGE ? 0 : off + STAGE;
            read(F[0], smem + off, 0);
        }
        if (whole) mma(F[1]);
        if constexpr (EPI == 2) {
            if ((q + 1) % spb == 0) { /* a K block ends: add its sum, start the next from zero */
                end_block(q + 1 == spb, q + 1 == nst);
            }
        }
    }

    if constexpr (EPI == 2) return; /* C is not touched */
    if constexpr (EPI == 1) {
        /* argmax partials: per row, the best (score + bias, lowest column) over this wavefront's
         * columns below keys_n, as one packed key per (row, column tile, wavefront column) */
        unsigned long long best[TI];
#pragma unroll
        for (int i = 0; i < TI; ++i) best[i] = 0;
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const u32 col = c0 + wn * WTN + 16 * j + 4 * fg + e;
                const bool ok = col < a.keys_n;
                const float bj = a.bias ? a.bias[col] : 0.0f;
#pragma unroll
                for (int i = 0; i < TI; ++i) {
                    const unsigned long long k = ok ? dec_key(acc[i][j][e] + bj, col) : 0ull;
                    best[i] = k > best[i] ? k : best[i];
                }
            }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            unsigned long long k = best[i];
#pragma unroll
            for (int msk = 16; msk < 64; msk <<= 1) {
                const unsigned long long o = shfl_xor_u64(k, msk);
                k = o > k ? o : k;
            }
            if (fg == 0 && row0 + 16 * i < M) a.keys[(u64)(row0 + 16 * i) * a.keys_ld + tn * WGN + wn] = k;
        }
        return;
    }

    constexpr int TO = GLU ? TJ / 2 : TJ;
    const u32 col0 = c0 + (GLU ? wn * (WTN / 2) : wn * WTN) + 4 * fg;
    floatx4 ba[TO] = {}, bb[TO] = {};
    if (a.bias)
#pragma unroll
        for (int j = 0; j < TO; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ba[j][e] = a.bias[col0 + 16 * j + e];
                if (GLU) bb[j][e] = a.bias[col0 + 16 * j + e + a.N / 2];
            }
    /* the four outputs of tile (i, j) */
    auto value = [&](int i, int j) {
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (GLU) {
                v[e] = (acc[i][j][e] + ba[j][e]) * sigmoid_f(acc[i][j + TJ / 2][e] + bb[j][e]) * a.alpha;
            } else {
                v[e] = acc[i][j][e] + ba[j][e];
                if (a.act == NK_ACT_SILU) v[e] = silu_f(v[e]);
                else if (a.act == NK_ACT_RELU) v[e] = fmaxf(v[e], 0.0f);
                v[e] *= a.alpha;
            }
        }
        return v;
    };
    if constexpr (OS) {
        /* split rows of nout values: hi at C2[row * ldc + n], lo at + nout (8-byte aligned: the host
         * checks C2 and ldc, and every tile divides nout into multiples of 4 columns) */
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TO; ++j) {
                const floatx4 v = value(i, j);
                if (row0 + 16 * i < M)
                    store_split4(a.C2 + (u64)(row0 + 16 * i) * a.ldc, nout, col0 + 16 * j, make_float4(v[0], v[1], v[2], v[3]));
            }
        return;
    }
    /* f32 rows, through the row map; four columns at once where C's rows are 16-byte aligned */
    const bool vec = a.ldc % 4 == 0 && ((size_t)a.C & 15) == 0;
    u32 orow[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const u32 r = min(row0 + 16 * i, M - 1);
        orow[i] = a.crow ? (u32)a.crow[r] : r;
    }
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        float *const dst = a.C + (u64)orow[i] * a.ldc + col0;
        floatx4 cv[TO];
#pragma unroll
        for (int j = 0; j < TO; ++j) {
            cv[j] = (floatx4){ 0.f, 0.f, 0.f, 0.f };
            if (a.accumulate) {
                if (vec) cv[j] = *(const floatx4 *)(dst + 16 * j);
                else
#pragma unroll
                    for (int e = 0; e < 4; ++e) cv[j][e] = dst[16 * j + e];
            }
        }
#pragma unroll
        for (int j = 0; j < TO; ++j) {
            floatx4 v = value(i, j);
            if (a.accumulate) v = cv[j] + v;
            if (row0 + 16 * i >= M) continue;
            if (vec) *(floatx4 *)(dst + 16 * j) = v;
            else
#pragma unroll
                for (int e = 0; e < 4; ++e) dst[16 * j + e] = v[e];
        }
    }
}

/* Tiles and ring depths.  128x256 and 96x256 take a CU each; which of the two leaves fewer CUs idle
 * depends on the rows (1300 rows, FF up in one round of 224 tiles of 96x256 29.9 us, 176 of 128x256 34.9; 3584
 * rows, QKV 49.1 against 57.1, FF up 77.3 against 69).  64x128 and 64x64 fit two workgroups on a CU (2 x 64 KB, 2 x 72 KB of its
 * 160 KB of LDS): one's MFMAs run while the other waits at its barrier, the better choice once there
 * are more than 256 workgroups.  64x128d (four stages), 32x64 and 32x32 take a CU each, with nearly
 * all of a 1024-column K loop's loads in flight at once: for launches of up to 256 workgroups, whose
 * time is the latency of one.  At 18 rows FF up takes 6.6 us on 32x32 tiles, 7.3 on 32x64, 8.7 on
 * 64x64; at 448 rows 13.8 on 64x128d (eight computing wavefronts, which share the epilogue; with four 15.0), 14.5
 * on 64x64, 16.8 on 64x128.  The host chooses by a cost per
 * round (mx_tile in csrc/host/nk.c).  Second launch bound: wavefronts per SIMD where two workgroups
 * fit a CU's LDS. */
#define GEMM_MX(NAME, BM, BN, WGM, WGN, PW, NS, GLU, EPI, AS, OS)                                         \
    extern "C" __global__ __launch_bounds__(64 * (WGM * WGN + PW),                                        \
                                            NS * (BM * 2 + BN) * 128 <= 81920 ? (WGM * WGN + PW) / 2 : 1) \
    void NAME(const NkGemmArgs a) {                                                                       \
        __shared__ uint4 ring_mem[NS * (BM * 2 + BN) * 8];                                                \
        mx_impl<BM, BN, WGM, WGN, PW, NS, GLU, EPI, AS, OS>(a, (lds_char_t *)ring_mem);                   \
    }
/* one tile in the forms of split-row A: f32 outputs, split-row outputs, GLU, residual update */
#define GEMM_MX_S(T, BM, BN, WGM, WGN, PW, NS)                                                            \
    GEMM_MX(gemm_mx##T##_s, BM, BN, WGM, WGN, PW, NS, false, 0, true, false)                              \
    GEMM_MX(gemm_mx##T##_s_so, BM, BN, WGM, WGN, PW, NS, false, 0, true, true)                            \
    GEMM_MX(gemm_mx##T##_acc_s, BM, BN, WGM, WGN, PW, NS, false, 2, true, false)
#define GEMM_MX_SG(T, BM, BN, WGM, WGN, PW, NS) GEMM_MX(gemm_mx##T##_glu_s, BM, BN, WGM, WGN, PW, NS, true, 0, true, false)
/* a residual update whose workgroups run all K blocks */
#define GEMM_MX_U(T, BM, BN, WGM, WGN, PW, NS)                                                            \
    extern "C" __global__ __launch_bounds__(64 * (WGM * WGN + PW)) void gemm_mx##T##_acc_s(const NkGemmArgs a) { \
        __shared__ uint4 ring_mem[NS * (BM * 2 + BN) * 8];                                                \
        mx_impl<BM, BN, WGM, WGN, PW, NS, false, 2, true, false, true>(a, (lds_char_t *)ring_mem);        \
    }
/* and of f32 A */
#define GEMM_MX_F(T, BM, BN, WGM, WGN, PW, NS)                                                            \
    GEMM_MX(gemm_mx##T, BM, BN, WGM, WGN, PW, NS, false, 0, false, false)                                 \
    GEMM_MX(gemm_mx##T##_so, BM, BN, WGM, WGN, PW, NS, false, 0, false, true)                             \
    GEMM_MX(gemm_mx##T##_acc, BM, BN, WGM, WGN, PW, NS, false, 2, false, false)
#define GEMM_MX_FG(T, BM, BN, WGM, WGN, PW, NS) GEMM_MX(gemm_mx##T##_glu, BM, BN, WGM, WGN, PW, NS, true, 0, false, false)
#define GEMM_MX_SS(...) GEMM_MX_S(__VA_ARGS__) GEMM_MX_SG(__VA_ARGS__)
#define GEMM_MX_FF(...) GEMM_MX_F(__VA_ARGS__) GEMM_MX_FG(__VA_ARGS__)
GEMM_MX_SS(128x256, 128, 256, 2, 4, 0, 2)
GEMM_MX_SS(96x256, 96, 256, 2, 4, 0, 2)
GEMM_MX_SS(64x128, 64, 128, 2, 2, 4, 2)
GEMM_MX_S(64x128d, 64, 128, 2, 4, 4, 4)
GEMM_MX_SG(64x128d, 64, 128, 2, 2, 4, 4)
GEMM_MX_SS(64x64, 64, 64, 2, 2, 4, 3)
GEMM_MX_SS(32x64, 32, 64, 2, 2, 4, 9)
GEMM_MX_S(32x32, 32, 32, 2, 2, 4, 12)
GEMM_MX_U(64x128u, 64, 128, 2, 2, 0, 2)
GEMM_MX_FF(64x128, 64, 128, 2, 2, 4, 2)
GEMM_MX_FF(64x64, 64, 64, 2, 2, 4, 3)
GEMM_MX_FF(32x64, 32, 64, 2, 2, 4, 9)
GEMM_MX_F(32x32, 32, 32, 2, 2, 4, 12)
/* residual updates on f32 rows: with 64x128 a wavefront's split A, its sums and the partial row it reads
 * back at a block's end exceed the 128 registers that two workgroups per CU leave; eight computing
 * wavefronts on 128x128, one workgroup per CU, have 170 and half the staged weights per MFMA (3584 x 2048,
 * K 4096, with the fold: 203 -> 175 us; 1792 x 1024, K 1024: 24.2 -> 22.5) */
GEMM_MX(gemm_mx128x128_acc, 128, 128, 4, 2, 4, 3, false, 2, false, false)
/* joint scores -> argmax partials (keys), 64x64 tiles: two keys per row per column tile */
GEMM_MX(gemm_mx64x64_argmax, 64, 64, 2, 2, 4, 3, false, 1, false, false)
