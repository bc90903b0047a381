/* Streaming-chunk kernels for gfx950 besides the GEMMs and the per-row kernels of nk_seq.hip:
 * the subsampling convs, copies, cache compaction, and the
 * RNNT decoder's LSTM cell and joint argmax.  Each states the reference kernel it replaces. */
#include "nk_common.h"

/* The two stride-2 3x3 convolutions of the subsampling, same causal padding (2 rows/columns
 * before, reference src/kernels.metal:411-454).  Workgroup = one output row t1 and 8 output
 * columns f1 (grid.x = T1 * ceil(F1/8), grid.y = windows of one size back to back, X and Y strides
 * xs / ys); thread = output channel, holding its 9 taps and bias in registers for the 8 columns.
 * Each output sums bias, then taps in (kh, kw) order. */
/* 1 input channel -> C channels + ReLU: X [T][F] -> Y [T1][F1][C] */
extern "C" __global__ __launch_bounds__(256) void conv2d_c1_s2_relu(NkConvArgs a) {
    const u32 nfb = (a.F1 + a.fb - 1) / a.fb;
    const u32 t1 = blockIdx.x / nfb, f0 = (blockIdx.x % nfb) * a.fb;
    const float *X = a.X + (u64)blockIdx.y * a.xs;
    float *Y = a.Y + (u64)blockIdx.y * a.ys;
    const u32 fe = min(f0 + a.fb, a.F1);
    for (u32 o = threadIdx.x; o < a.C; o += 256) {
        float w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = a.W[o * 9 + k];
        const float bo = a.bias[o];
        for (u32 f1 = f0; f1 < fe; ++f1) {
            float acc = bo;
#pragma unroll
            for (int kh = 0; kh < 3; ++kh) {
                const int ti = (int)(2 * t1 + kh) - 2;
                if (ti < 0 || ti >= (int)a.T) continue;
#pragma unroll
                for (int kw = 0; kw < 3; ++kw) {
                    const int fi = (int)(2 * f1 + kw) - 2;
                    if (fi < 0 || fi >= (int)a.F) continue;
                    acc += w[kh * 3 + kw] * X[(u64)ti * a.F + fi];
                }
            }
            Y[((u64)t1 * a.F1 + f1) * a.C + o] = fmaxf(acc, 0.0f);
        }
    }
}

/* depthwise, + bias, no activation: X [T][F][C] -> Y [T1][F1][C] */
extern "C" __global__ __launch_bounds__(256) void dwconv2d_s2(NkConvArgs a) {
    const u32 nfb = (a.F1 + a.fb - 1) / a.fb;
    const u32 t1 = blockIdx.x / nfb, f0 = (blockIdx.x % nfb) * a.fb;
    const float *X = a.X + (u64)blockIdx.y * a.xs;
    float *Y = a.Y + (u64)blockIdx.y * a.ys;
    const u32 fe = min(f0 + a.fb, a.F1);
    for (u32 c = threadIdx.x; c < a.C; c += 256) {
        float w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = a.W[c * 9 + k];
        const float bc = a.bias[c];
        for (u32 f1 = f0; f1 < fe; ++f1) {
            float acc = bc;
#pragma unroll
            for (int kh = 0; kh < 3; ++kh) {
                const int ti = (int)(2 * t1 + kh) - 2;
                if (ti < 0 || ti >= (int)a.T) continue;
#pragma unroll
                for (int kw = 0; kw < 3; ++kw) {
                    const int fi = (int)(2 * f1 + kw) - 2;
                    if (fi < 0 || fi >= (int)a.F) continue;
                    acc += w[kh * 3 + kw] * X[((u64)ti * a.F + fi) * a.C + c];
                }
            }
            Y[((u64)t1 * a.F1 + f1) * a.C + c] = acc;
        }
    }
}

/* The same, four channels per thread (C / 4 divides 256, 16-byte aligned rows): a thread computes DW2_FB
 * neighbouring outputs of one row, whose 9 input columns x 3 rows it loads at once (two new columns
 * per output instead of three, one memory round trip per thread; the taps come through LDS, where a
 * thread's 36 are nine 16-byte reads).  A tap outside X is added as a
 * product with zero, which changes nothing for a finite weight; outputs with a NaN among them are
 * computed again skipping it, as dwconv2d_s2 does.
 * 64 windows of 19 x 33 x 256: 32.1 -> 13.3 us (52 MB read and written: 10.7 at the rate of a copy),
 * 256 windows 120 -> 44 us. */
#define DW2_FB 4
/* output (t1, f1) of channels c .. c + 3, tap by tap; X: the window's channel c */
__device__ __forceinline__ floatx4 dw2_skipping(const NkConvArgs &a, const float *X, u32 c, u32 t1, u32 f1) {
    floatx4 acc = *(const floatx4 *)(a.bias + c);
#pragma unroll 1 /* rare: few registers and instructions */
    for (u32 k = 0; k < 9; ++k) {
        const int ti = (int)(2 * t1 + k / 3) - 2, fi = (int)(2 * f1 + k % 3) - 2;
        if (ti < 0 || ti >= (int)a.T || fi < 0 || fi >= (int)a.F) continue;
        const floatx4 v = *(const floatx4 *)(X + ((u64)ti * a.F + fi) * a.C);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += a.W[(c + e) * 9 + k] * v[e];
    }
    return acc;
}
extern "C" __global__ __launch_bounds__(256) void dwconv2d_s2_v4(NkConvArgs a) {
    __shared__ floatx4 taps[1024 * 9 / 4];
    const u32 C4 = a.C / 4, tid = threadIdx.x, per = 256 / C4;
    const u32 nfb = (a.F1 + DW2_FB - 1) / DW2_FB, seg = blockIdx.x * per + tid / C4;
    const u32 t1 = seg / nfb, f0 = (seg % nfb) * DW2_FB, c = 4 * (tid % C4);
    const float *X = a.X + (u64)blockIdx.y * a.xs + c;
    for (u32 i = tid; i < a.C * 9 / 4; i += 256) taps[i] = ((const floatx4 *)a.W)[i];
    const bool in = t1 < a.T1;
    floatx4 x[3][2 * DW2_FB + 1];
#pragma unroll
    for (int kh = 0; kh < 3; ++kh) {
        const int ti = (int)(2 * t1 + kh) - 2;
        const bool row = in && ti >= 0 && ti < (int)a.T;
#pragma unroll
        for (int k = 0; k < 2 * DW2_FB + 1; ++k) {
            const int fi = (int)(2 * f0 + k) - 2;
            const bool ok = row && fi >= 0 && fi < (int)a.F;
            const floatx4 v = *(const floatx4 *)(X + (ok ? ((u64)ti * a.F + fi) * a.C : 0));
            x[kh][k] = ok ? v : (floatx4){ 0.f, 0.f, 0.f, 0.f };
        }
    }
    const floatx4 bias = *(const floatx4 *)(a.bias + c);
    __syncthreads();
    if (!in) return;
    floatx4 w[9]; /* channel e, tap k is element 9 e + k */
#pragma unroll
    for (int k = 0; k < 9; ++k) w[k] = taps[(c / 4) * 9 + k];
    float *Y = a.Y + (u64)blockIdx.y * a.ys + ((u64)t1 * a.F1 + f0) * a.C + c;
    float sum = 0.0f;
#pragma unroll
    for (int f = 0; f < DW2_FB; ++f) {
        if (f0 + f >= a.F1) break;
        floatx4 acc = bias;
#pragma unroll
        for (int k = 0; k < 9; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += w[(9 * e + k) / 4][(9 * e + k) % 4] * x[k / 3][2 * f + k % 3][e];
        *(floatx4 *)(Y + (u64)f * a.C) = acc;
        sum += (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
    if (sum != sum) /* a NaN among them, perhaps from a weight times a position outside X */
#pragma unroll 1
        for (u32 f = 0; f < DW2_FB && f0 + f < a.F1; ++f) *(floatx4 *)(Y + (u64)f * a.C) = dw2_skipping(a, X, c, t1, f0 + f);
}

/* conv 0 (1 -> C channels + ReLU) followed by conv 2 (depthwise, + bias) without storing conv 0's
 * output: X [T][F] -> Y [T2][F2][C].  Workgroup = one output row t2 and fb output columns of one
 * window; thread = channel.  The seven X rows the output row reads (4 t2 - 6 .. 4 t2) are staged
 * in LDS.  Every conv 0 value is computed exactly as conv2d_c1_s2_relu computes it (bias, then the
 * taps in (kh, kw) order, taps outside X skipped, ReLU) and every output exactly as dwconv2d_s2
 * computes it (bias, then the taps in order, positions outside conv 0's T1 x F1 skipped), so the
 * result equals the two kernels' bit for bit.  A skipped tap is added here as a product with zero,
 * which changes nothing for a finite weight; a channel with an infinite or NaN weight is computed
 * again by a loop that skips.
 *
 * Bound by its 63 multiply-adds per output (17 us for 64 windows of 72 rows at the full vector rate), so
 * everything else is kept out of the loop: the mel rows lie in LDS with zeros around them, so no tap
 * is tested; a thread walks its columns left to right and reads the four new mel columns of each
 * output as one 16-byte broadcast per row (seven LDS reads where every column was read by itself, 49),
 * and the conv 0 column 2 f2 of output f2, which is column 2 (f2 + 1) - 2 of the next, is kept.
 * Positions outside conv 0 are masked, not branched around.  One window of 72 rows 8.4 -> 4.2 us, 64
 * windows 73 -> 31.4, 256 windows 216 -> 90 (0.12, 0.9 and 1 of these for the test of the weights and its
 * loop). */
#define CONV02_PAD 7 /* LDS index of mel column 0: the four new columns of output f2 start at 4 f2 + 4 */
#define CONV02_LDW (NK_CONV02_FMAX + 16)
/* outputs f0 .. fe - 1 of row t2, channel c, tap by tap */
__device__ __forceinline__ void conv02_skipping(const NkConv02Args &a, const float (*xs)[CONV02_LDW], u32 c, u32 t2, u32 f0,
                                             u32 fe, float *Y) {
#pragma unroll 1 /* rare: few registers and instructions */
    for (u32 f2 = f0; f2 < fe; ++f2) {
        float acc = a.b2[c];
#pragma unroll 1
        for (u32 k2 = 0; k2 < 9; ++k2) {
            const int t1 = (int)(2 * t2 + k2 / 3) - 2, f1 = (int)(2 * f2 + k2 % 3) - 2;
            if (t1 < 0 || t1 >= (int)a.T1 || f1 < 0 || f1 >= (int)a.F1) continue;
            float v = a.b0[c];
#pragma unroll 1
            for (u32 k = 0; k < 9; ++k) {
                const int ti = 2 * t1 + (int)(k / 3) - 2, fi = 2 * f1 + (int)(k % 3) - 2;
                if (ti < 0 || ti >= (int)a.T || fi < 0 || fi >= (int)a.F) continue;
                v += a.W0[c * 9 + k] * xs[2 * (k2 / 3) + k / 3][fi + CONV02_PAD];
            }
            acc += a.W2[c * 9 + k2] * fmaxf(v, 0.0f);
        }
        Y[((u64)t2 * a.F2 + f2) * a.C + c] = acc;
    }
}
extern "C" __global__ __launch_bounds__(256) void conv2d_c1_dw_s2(NkConv02Args a) {
    constexpr u32 LDW = CONV02_LDW;
    __shared__ __attribute__((aligned(16))) float xs[7][LDW];
    const u32 nfb = (a.F2 + a.fb - 1) / a.fb;
    const u32 t2 = blockIdx.x / nfb, f0 = (blockIdx.x % nfb) * a.fb;
    const float *X = a.X + (u64)blockIdx.y * a.xs;
    float *Y = a.Y + (u64)blockIdx.y * a.ys;
    const u32 fe = min(f0 + a.fb, a.F2);
    const int ti0 = 4 * (int)t2 - 6; /* X row of LDS row 0 */
    /* the LDS columns this workgroup's outputs read */
    const u32 i0 = min(4 * f0, LDW - 4), iw = min(4 * fe + 4, LDW) - i0;
    for (u32 i = threadIdx.x; i < 7 * iw; i += 256) {
        const u32 r = i / iw, k = i0 + i % iw;
        const int ti = ti0 + (int)r, col = (int)k - CONV02_PAD;
        xs[r][k] = ti >= 0 && ti < (int)a.T && col >= 0 && col < (int)a.F ? X[(u64)ti * a.F + col] : 0.0f;
    }
    __syncthreads();
    u32 row_in[3]; /* all ones for the conv 0 rows 2 t2 - 2 .. 2 t2 that exist */
#pragma unroll
    for (int k = 0; k < 3; ++k) row_in[k] = (u32)(2 * (int)t2 + k - 2) < a.T1 ? ~0u : 0u;
    for (u32 c = threadIdx.x; c < a.C; c += 256) {
        float w0[9], w2[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) { w0[k] = a.W0[c * 9 + k]; w2[k] = a.W2[c * 9 + k]; }
        const float bias0 = a.b0[c], bias2 = a.b2[c];
        float odd[3] = { 0.f, 0.f, 0.f }; /* 0, or NaN with a weight that is not finite */
#pragma unroll
        for (int k = 0; k < 9; ++k) odd[k % 3] += w0[k] * 0.0f + w2[k] * 0.0f;
        if (odd[0] + odd[1] + odd[2] != 0.0f) {
            conv02_skipping(a, xs, c, t2, f0, fe, Y);
            continue;
        }
        /* mel columns 4 f2 - 6 .. 4 f2 of the seven rows; conv 0's column 2 f2 - 2 of output f2 */
        float xv[7][7], keep[3];
        /* conv 0 at row 2 t2 + kh2 - 2, column f1: mel row 2 kh2 + kh, columns q .. q + 2 of xv */
        auto conv0 = [&](const int kh2, const int q, const u32 f1) -> float {
            float acc = bias0;
#pragma unroll
            for (int kh = 0; kh < 3; ++kh)
#pragma unroll
                for (int kw = 0; kw < 3; ++kw) acc += w0[kh * 3 + kw] * xv[2 * kh2 + kh][q + kw];
            const u32 in = row_in[kh2] & (f1 < a.F1 ? ~0u : 0u); /* uniform: a mask, not a branch */
            return __uint_as_float(__float_as_uint(fmaxf(acc, 0.0f)) & in);
        };
#pragma unroll
        for (int r = 0; r < 7; ++r)
#pragma unroll
            for (int q = 0; q < 3; ++q) xv[r][4 + q] = xs[r][min(4 * f0 + 1 + q, LDW - 1)];
#pragma unroll
        for (int kh2 = 0; kh2 < 3; ++kh2) keep[kh2] = conv0(kh2, 4, 2 * f0 - 2);
        for (u32 f2 = f0; f2 < fe; ++f2) {
#pragma unroll
            for (int r = 0; r < 7; ++r) {
                const floatx4 n = *(const floatx4 *)&xs[r][min(4 * f2 + 4, LDW - 4)];
#pragma unroll
                for (int q = 0; q < 3; ++q) xv[r][q] = xv[r][4 + q];
#pragma unroll
                for (int q = 0; q < 4; ++q) xv[r][3 + q] = n[q];
            }
            float acc = bias2;
#pragma unroll
            for (int kh2 = 0; kh2 < 3; ++kh2) {
                const float v1 = conv0(kh2, 2, 2 * f2 - 1), v2 = conv0(kh2, 4, 2 * f2);
                acc += w2[kh2 * 3] * keep[kh2];
                acc += w2[kh2 * 3 + 1] * v1;
                acc += w2[kh2 * 3 + 2] * v2;
                keep[kh2] = v2;
            }
            Y[((u64)t2 * a.F2 + f2) * a.C + c] = acc;
        }
    }
}

/* Log-mel of one 512-sample frame per workgroup (reference src/mel.c:115-173, the host front end's
 * computation step for step): window, radix-2 decimation-in-time FFT in double (bit-reversed load,
 * nine stages of 256 butterflies, one per thread, with the host's twiddle table and operation
 * order), power in double rounded to float, each filter's sum over its bins in ascending order in
 * float, log(x + 2^-24).  Floating-point contraction is off, so the spectrum equals the host's. */
extern "C" __global__ __launch_bounds__(256) void mel_frames(const NkMelArgs a) {
#pragma clang fp contract(off)
    __shared__ double re[512], im[512];
    __shared__ float pw[257];
    const u32 f = blockIdx.x, t = threadIdx.x;
    const float *fr = a.span + a.tab[2 * f];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const u32 k = t + 256 * h, j = a.rev[k];
        re[j] = (double)(fr[k] * a.win[k]);
        im[j] = 0.0;
    }
    __syncthreads();
    for (u32 len = 2; len <= 512; len <<= 1) {
        const u32 hl = len >> 1, stride = 512 / len, k = t % hl, ia = (t / hl) * len + k, ib = ia + hl;
        const double wr = a.tw_re[k * stride], wi = a.tw_im[k * stride];
        const double br = re[ib], bi = im[ib], ar = re[ia], ai = im[ia];
        const double xr = br * wr - bi * wi, xi = br * wi + bi * wr;
        re[ib] = ar - xr;
        im[ib] = ai - xi;
        re[ia] = ar + xr;
        im[ia] = ai + xi;
        __syncthreads();
    }
    pw[t] = (float)(re[t] * re[t] + im[t] * im[t]);
    if (t == 0) pw[256] = (float)(re[256] * re[256] + im[256] * im[256]);
    __syncthreads();
    if (t < 128) {
        float acc = 0.0f;
        const float *w = a.fb + (u64)t * 257;
        for (int k = a.fb_lo[t]; k < a.fb_hi[t]; ++k) acc += w[k] * pw[k];
        a.out[(u64)(u32)a.tab[2 * f + 1] * 128 + t] = logf(acc + 5.9604644775390625e-08f);
    }
}

/* [T][F][C] -> [T][C*F] channel-major flatten (reference src/kernels.metal:456-462) of many rows: one
 * [F][C] row of a window per workgroup through LDS (F (C + 4) floats of at most NK_FLAT_LDS, C % 4 == 0,
 * 16-byte aligned), so that both the reads and the writes are whole lines; a thread's own elements
 * were C apart.  LDS rows are C + 4 floats, which spreads the reads along f over the banks.
 * 64 windows of 10 x 17 x 256: 9.9 -> 6.6 us, 256 windows 30.1 -> 16.2. */
extern "C" __global__ __launch_bounds__(256) void flatten_cf_t(const NkFlatArgs a) {
    __shared__ __attribute__((aligned(16))) float s[NK_FLAT_LDS];
    const u64 base = ((u64)blockIdx.y * a.T + blockIdx.x) * a.F * a.C;
    const u32 n4 = a.F * a.C / 4, C4 = a.C / 4;
    for (u32 i = threadIdx.x; i < n4; i += 256)
        *(floatx4 *)&s[(i / C4) * (a.C + 4) + 4 * (i % C4)] = *(const floatx4 *)(a.X + base + 4 * (u64)i);
    __syncthreads();
    for (u32 i = threadIdx.x; i < n4; i += 256) {
        u32 c = 4 * i / a.F, f = 4 * i - c * a.F;
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = s[f * (a.C + 4) + c];
            if (++f == a.F) { f = 0; ++c; }
        }
        *(floatx4 *)(a.Y + base + 4 * (u64)i) = v;
    }
}

/* The same, one thread per output element (reads gather, writes are coalesced). */
extern "C" __global__ __launch_bounds__(256) void flatten_cf(NkFlatArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x;
    const u64 total = (u64)a.T * a.C * a.F;
    if (idx >= total) return;
    a.X += (u64)blockIdx.y * total; /* grid.y: windows of the same size, back to back */
    a.Y += (u64)blockIdx.y * total;
    const u32 f = (u32)(idx % a.F), c = (u32)((idx / a.F) % a.C), t = (u32)(idx / ((u64)a.F * a.C));
    a.Y[idx] = a.X[((u64)t * a.F + f) * a.C + c];
}

extern "C" __global__ __launch_bounds__(256) void copy_f32(const NkCopyArgs a) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.n) a.dst[i] = a.src[i];
}

/* Pending residual update of the many-row GEMM (NkFoldArgs): one thread per 4 consecutive values
 * of a row, the parts added in order from zero, then C + alpha * sum. */
extern "C" __global__ __launch_bounds__(256) void resid_fold(const NkFoldArgs a) {
    const u32 n4 = a.N >> 2, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.M * n4) return;
    const u32 r = i / n4, c = 4 * (i % n4);
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
    for (u32 b = 0; b < a.nparts; ++b) {
        const float4 q = *(const float4 *)(a.P + ((u64)b * a.M + r) * a.N + c);
        t.x += q.x; t.y += q.y; t.z += q.z; t.w += q.w;
    }
    float4 *dst = (float4 *)(a.C + (u64)r * a.ldc + c);
    float4 v = *dst;
    v.x = v.x + t.x * a.alpha; v.y = v.y + t.y * a.alpha; v.z = v.z + t.z * a.alpha; v.w = v.w + t.w * a.alpha;
    *dst = v;
}

extern "C" __global__ __launch_bounds__(256) void fill_f32(const NkFillArgs a) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.n) a.dst[i] = a.value;
}

/* Epoch compaction of the per-layer caches in one launch (reference src/encoder.c:199-211 issues
 * one copy per layer and cache).  grid = (ceil(rows*cols/256), nbuf).  Source and destination rows
 * never overlap (the host checks src_row >= dst_row + rows). */
extern "C" __global__ __launch_bounds__(256) void compact_rows(const NkCompactArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (u64)a.rows * a.cols) return;
    float *b = a.base + (u64)blockIdx.y * a.stride;
    b[(u64)a.dst_row * a.cols + idx] = b[(u64)a.src_row * a.cols + idx];
}
/* The same copy 16 bytes per thread, when cols, the buffer stride and the base are multiples of 4
 * floats (every cache of the model: rows of 1024 or 3072 floats).  grid = (ceil(rows*cols/1024), nbuf). */
extern "C" __global__ __launch_bounds__(256) void compact_rows4(const NkCompactArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x, n4 = (u64)a.rows * a.cols / 4;
    if (idx >= n4) return;
    float4 *b = (float4 *)(a.base + (u64)blockIdx.y * a.stride);
    b[(u64)a.dst_row * (a.cols / 4) + idx] = b[(u64)a.src_row * (a.cols / 4) + idx];
}

/* State of a fresh stream (NkResetArgs); grid = (ceil(max(n, zn) / 256), nbuf + 1), the last y the
 * decoder's part.  One launch for the copies of a stream's reset: they were 27 small host-to-device
 * copies of zeros, each waited for (~8 us), 14 of the 51 ms of a pass that resets 64 streams. */
extern "C" __global__ __launch_bounds__(256) void stream_reset(const NkResetArgs a) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.y < a.nbuf) {
        if (i < a.n) a.base[blockIdx.y * a.stride + i] = 0.0f;
        return;
    }
    if (i < a.zn) {
        if (a.z0) a.z0[i] = 0.0f;
        if (a.z1) a.z1[i] = 0.0f;
    }
    if (i < a.words) a.st[i] = a.val[i];
}

/* Strided row copy: rows x cols floats from src (row stride src_ld) to dst (row stride dst_ld).
 * Used for the row select of the subsampled window and for activation dumps. */
extern "C" __global__ __launch_bounds__(256) void copy2d_f32(const NkCopy2dArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (u64)a.rows * a.cols) return;
    const u32 r = (u32)(idx / a.cols), c = (u32)(idx % a.cols);
    a.dst[(u64)r * a.dst_ld + c] = a.src[(u64)r * a.src_ld + c];
}

/* ---- batched streams ------------------------------------------------------------------------ */

/* dst[m] = src[map[m]] row gather (the batched row select of the subsampled windows) */
extern "C" __global__ __launch_bounds__(256) void gather_rows(const NkGatherArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (u64)a.rows * a.cols) return;
    const u32 m = (u32)(idx / a.cols), k = (u32)(idx % a.cols);
    a.dst[(u64)m * a.dst_ld + k] = a.src[(u64)(u32)a.map[m] * a.src_ld + k];
}

/* dst row map[m] = src row m (rows of `cols` floats; the map's targets are distinct) */
extern "C" __global__ __launch_bounds__(256) void scatter_rows(const NkGatherArgs a) {
    const u64 idx = (u64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (u64)a.rows * a.cols) return;
    const u32 m = (u32)(idx / a.cols), k = (u32)(idx % a.cols);
    a.dst[(u64)(u32)a.map[m] * a.dst_ld + k] = a.src[(u64)m * a.src_ld + k];
}

/* LSTM input rows [x | h] of the batched decoder (one thread per element; grid.y = row) */
extern "C" __global__ __launch_bounds__(256) void lstm_input_rows(const NkLstmInArgs a) {
    const u32 n = blockIdx.y, k = blockIdx.x * 256 + threadIdx.x;
    if (n >= a.n || k >= 2 * a.P) return;
    float v;
    if (k < a.P) {
        if (a.tok) {
            const int t = a.tok[n];
            v = (t < 0 || (u32)t == a.blank) ? 0.0f : bf2f(a.embed[(u64)t * a.P + k]);
        } else {
            v = a.xsrc[(u64)n * a.P + k];
        }
    } else {
        v = a.hc[(u64)(u32)a.hrow[n] * a.P + (k - a.P)];
    }
    a.A[(u64)n * 2 * a.P + k] = v;
}

/* LSTM cell on batched rows, reference src/kernels.metal:474-486 (c' = f*c + i*g, h' = o*tanh(c')) */
extern "C" __global__ __launch_bounds__(256) void lstm_cell_rows(const NkLstmRowsArgs a) {
    const u32 n = blockIdx.y, j = blockIdx.x * 256 + threadIdx.x;
    if (n >= a.n || j >= a.P) return;
    const float *gt = a.gates + (u64)n * 4 * a.P;
    const float ig = sigmoid_f(gt[j]), fg = sigmoid_f(gt[a.P + j]), gg = tanhf(gt[2 * a.P + j]), og = sigmoid_f(gt[3 * a.P + j]);
    const float c = fg * a.hc[(u64)(u32)a.crow_in[n] * a.P + j] + ig * gg;
    const float h = og * tanhf(c);
    a.hc[(u64)(u32)a.crow_out[n] * a.P + j] = c;
    a.hc[(u64)(u32)a.hrow_out[n] * a.P + j] = h;
    a.hout[(u64)n * a.P + j] = h;
}

/* joint input rows relu(enc + pred), reference src/kernels.metal:488-519 (the r vector) */
extern "C" __global__ __launch_bounds__(256) void joint_in_rows(const NkJointInArgs a) {
    const u32 r = blockIdx.y, k = blockIdx.x * 256 + threadIdx.x;
    if (r >= a.rows || k >= a.J) return;
    a.jin[(u64)r * a.J + k] = fmaxf(a.enc[(u64)(u32)a.erow[r] * a.J + k] + a.pred[(u64)(u32)a.prow[r] * a.J + k], 0.0f);
}

/* argmax of each row of joint logits, lowest index on ties (src/kernels.metal:521-550) */
extern "C" __global__ __launch_bounds__(256) void argmax_rows(const NkArgmaxRowsArgs a) {
    __shared__ float bv[256];
    __shared__ int bi[256];
    const u32 r = blockIdx.x, tid = threadIdx.x;
    const float *x = a.logits + (u64)r * a.ld;
    float best = -INFINITY;
    int bidx = 0x7fffffff;
    for (u32 n = tid; n < a.V; n += 256) {
        const float v = x[n];
        if (v > best || (v == best && (int)n < bidx)) { best = v; bidx = (int)n; }
    }
    bv[tid] = best;
    bi[tid] = bidx;
    __syncthreads();
    for (u32 st = 128; st > 0; st >>= 1) {
        if (tid < st) {
            const float ov = bv[tid + st];
            const int oi = bi[tid + st];
            if (ov > bv[tid] || (ov == bv[tid] && oi < bi[tid])) { bv[tid] = ov; bi[tid] = oi; }
        }
        __syncthreads();
    }
    if (tid == 0) {
        a.out[2 * r] = bi[0];
        a.out[2 * r + 1] = __float_as_int(bv[0]);
    }
}
