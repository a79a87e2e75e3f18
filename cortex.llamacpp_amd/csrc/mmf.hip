// mmf.hip — batched contraction against F16 weight tensors on the matrix cores (ggml_mul_mat with an f16 src0: the CPU path rounds the activations to f16 and
// takes vec_dot_f16, f32 accumulation; SURVEY.md §8a row a10 for files that keep their projections in f16 — the reference's embedding smoke model is one, Makefile:6).
//
//   Y[t][n] (+ resid[t][n]) = sum_k W[n][k] * f16(X[t][k])
//
// Both operands are K-contiguous rows, which is exactly the register layout of v_mfma_f32_32x32x16_f16 (lane = (row m, k-group kg): eight consecutive k), so
// neither goes through LDS: a wave owns a 64 x 64 (weight rows x tokens) tile as 2 x 2 MFMA tiles and reads its A rows as 16-byte loads and its B rows as two
// float4 loads converted to halfs in registers; the four waves of a workgroup form a 128 x 128 tile and share their rows through the caches.  The products are
// exact in f32 and summed in f32 by the matrix pipe (the CPU sums lane-wise partials of the same products: equal up to f32 re-association).
// One wave per (row, token) - mmv_float_kernel, misc.hip - stays the path for single tokens and for f32 tensors.
#include <cstdlib>

#include "kernels.h"

namespace mi355 {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// WT = 32 x 32 tiles a wave holds per side: 2 -> a workgroup covers 128 x 128 outputs, 1 -> 64 x 64 (four times the workgroups: shapes whose 128-tiles would leave
// most of the 256 CUs idle - the LLaVA tower's 577 x 1024 projections are 40 of them).  Every output is the same chain of matrix-core steps over k either way.
// XH: the activations arrive as f16 already (launch_f32_to_f16 - the same rounding, done once per row instead of once per workgroup column that reads it).
// Epilogue: y = resid + (acc + bias) * scale, each part optional (bias per output column, then the scale, then the residual row: the order of the separate
// bias / scale / add launches it replaces).
template <int WT, bool XH>
__global__ __launch_bounds__(256) void mmf16_kernel(const _Float16 *W, int N, int K, const void *Xv, int T, float *Y, int ldy, const float *resid, const float *bias,
                                                    float scale, int do_scale) {
    const float *X = reinterpret_cast<const float *>(Xv);
    const _Float16 *Xh = reinterpret_cast<const _Float16 *>(Xv);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 31, kg = lane >> 5;
    const int n0 = blockIdx.x * (64 * WT) + (wave & 1) * (32 * WT), t0 = blockIdx.y * (64 * WT) + (wave >> 1) * (32 * WT);
    if (n0 >= N || t0 >= T) return;                             // (wave-uniform)
    const _Float16 *wr[WT], *xh[WT];
    const float *xr[WT];
#pragma unroll
    for (int i = 0; i < WT; i++) {
        const int n = n0 + 32 * i + m, t = t0 + 32 * i + m;     // rows past the end read the last row; their results are never stored
        wr[i] = W + (size_t)(n < N ? n : N - 1) * K + 8 * kg;
        xr[i] = X + (size_t)(t < T ? t : T - 1) * K + 8 * kg;
        xh[i] = Xh + (size_t)(t < T ? t : T - 1) * K + 8 * kg;
    }
    f32x16 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
#pragma unroll 2
    for (int k0 = 0; k0 < K; k0 += 16) {
        f16x8 a[WT], b[WT];
#pragma unroll
        for (int i = 0; i < WT; i++) {
            a[i] = *reinterpret_cast<const f16x8 *>(wr[i] + k0);
            if constexpr (XH) b[i] = *reinterpret_cast<const f16x8 *>(xh[i] + k0);
            else {
                const f32x4 x0 = *reinterpret_cast<const f32x4 *>(xr[i] + k0), x1 = *reinterpret_cast<const f32x4 *>(xr[i] + k0 + 4);
                b[i][0] = (_Float16)x0.x; b[i][1] = (_Float16)x0.y; b[i][2] = (_Float16)x0.z; b[i][3] = (_Float16)x0.w;
                b[i][4] = (_Float16)x1.x; b[i][5] = (_Float16)x1.y; b[i][6] = (_Float16)x1.z; b[i][7] = (_Float16)x1.w;
            }
        }
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < WT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    // register r of a lane: weight row (r & 3) + 8 (r >> 2) + 4 kg of the tile, token = lane & 31: four consecutive rows per 16-byte store
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++) {
            const int t = t0 + 32 * j + m;
            if (t >= T) continue;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n = n0 + 32 * i + 8 * q + 4 * kg;
                float *dst = Y + (size_t)t * ldy + n;
                const float *rs = resid ? resid + (size_t)t * ldy + n : nullptr;
                float r[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    r[e] = acc[i][j][4 * q + e];
                    if (bias && n + e < N) r[e] = r[e] + bias[n + e];
                    if (do_scale) r[e] = r[e] * scale;
                }
                if (n + 3 < N && (ldy & 3) == 0) {
                    f32x4 v = {r[0], r[1], r[2], r[3]};
                    if (rs) { const f32x4 r4 = *reinterpret_cast<const f32x4 *>(rs); v.x = r4.x + v.x; v.y = r4.y + v.y; v.z = r4.z + v.z; v.w = r4.w + v.w; }
                    *reinterpret_cast<f32x4 *>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) if (n + e < N) dst[e] = rs ? rs[e] + r[e] : r[e];
                }
            }
        }
}

}  // namespace

bool mmf16_applicable(int type, int n_rows, int K, int T, const void *W, const void *x, const void *y) {
    return type == T_F16 && T >= 8 && n_rows >= 32 && (K % 16) == 0 && ((reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
}

namespace {
// The f16 x f16 product staged through LDS: 64 x 64 outputs per workgroup, 64 halves of k per stage (one 128-byte line of every row: eight lanes fetch a row's
// line together, where the direct kernel's lanes each fetch 16 bytes of a different row - 32 lines, on few L2 channels when the row stride is a power of two),
// double-buffered; a wave owns 32 x 32 outputs and reads its two fragments per matrix-core step from rows padded to 144 bytes (conflict-free 16-byte reads).
// The same chain of matrix-core steps over k as mmf16_kernel: the results agree bit for bit.
__global__ __launch_bounds__(256) void mmf16_lds_kernel(const _Float16 *__restrict__ W, int N, int K, const _Float16 *__restrict__ X, int T, float *Y, int ldy,
                                                        const float *resid, const float *bias, float scale, int do_scale) {
    constexpr int BK = 64, LDR = 72;                            // halves per stage, padded row length (144 bytes)
    __shared__ _Float16 sA[2][64 * LDR], sB[2][64 * LDR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 31, kg = lane >> 5;
    const int n0 = blockIdx.x * 64, t0 = blockIdx.y * 64;
    const int lr = tid >> 3, lc = tid & 7;                      // loader: rows lr and lr + 32 of both tiles, 16-byte column lc
    const _Float16 *gw[2], *gx[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int n = n0 + lr + 32 * i, t = t0 + lr + 32 * i;   // rows past the end read the last row; their results are never stored
        gw[i] = W + (size_t)(n < N ? n : N - 1) * K + 8 * lc;
        gx[i] = X + (size_t)(t < T ? t : T - 1) * K + 8 * lc;
    }
    // PD stages of k are on their way at any time (registers), one is in LDS being used, the next is being written to the other LDS buffer: a stage's matrix
    // work is 4 steps (tens of ns) against a memory round trip of a microsecond, and the 577 x 1024 products have only 160 workgroups to overlap with
    constexpr int PD = 4;
    f16x8 ra[PD][2], rb[PD][2];
    // (no branch and no select around a load: either would make the compiler drain every load in flight where the paths join.  A piece past K - the last stage
    // of a K that is not a multiple of 64, and the stages requested past the end - is read from the row's last 16 bytes instead and never multiplied)
    auto fetch = [&](f16x8 (&a2)[2], f16x8 (&b2)[2], int k0) {
        const int k = k0 + 8 * lc < K ? k0 : K - 8 - 8 * lc;
#pragma unroll
        for (int i = 0; i < 2; i++) { a2[i] = *reinterpret_cast<const f16x8 *>(gw[i] + k); b2[i] = *reinterpret_cast<const f16x8 *>(gx[i] + k); }
    };
    auto put = [&](const f16x8 (&a2)[2], const f16x8 (&b2)[2], int buf) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            *reinterpret_cast<f16x8 *>(&sA[buf][(lr + 32 * i) * LDR + 8 * lc]) = a2[i];
            *reinterpret_cast<f16x8 *>(&sB[buf][(lr + 32 * i) * LDR + 8 * lc]) = b2[i];
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    const int ar = ((wave & 1) * 32 + m) * LDR + 8 * kg, br = ((wave >> 1) * 32 + m) * LDR + 8 * kg;
    const int nst = (K + BK - 1) / BK;
#pragma unroll
    for (int u = 0; u < PD; u++) fetch(ra[u], rb[u], u * BK);
    put(ra[0], rb[0], 0);
    __syncthreads();
    for (int st = 0; st < nst; st += PD) {
#pragma unroll
        for (int u = 0; u < PD; u++) {
            const int cur = st + u, buf = u & 1;
            if (cur >= nst) break;
            fetch(ra[u], rb[u], (cur + PD) * BK);               // slot u went to LDS a step ago: refill it PD stages ahead
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) {
                if (cur * BK + 16 * s4 >= K) break;
                const f16x8 a = *reinterpret_cast<const f16x8 *>(&sA[buf][ar + 16 * s4]), b = *reinterpret_cast<const f16x8 *>(&sB[buf][br + 16 * s4]);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
            }
            if (cur + 1 < nst) put(ra[(u + 1) % PD], rb[(u + 1) % PD], buf ^ 1);
            __syncthreads();
        }
    }
    // register r of a lane: weight row (r & 3) + 8 (r >> 2) + 4 kg of the wave's tile, token = lane & 31 (as in mmf16_kernel)
    const int t = t0 + (wave >> 1) * 32 + m;
    if (t >= T) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int n = n0 + (wave & 1) * 32 + 8 * q + 4 * kg;
        float *dst = Y + (size_t)t * ldy + n;
        const float *rs = resid ? resid + (size_t)t * ldy + n : nullptr;
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            r[e] = acc[4 * q + e];
            if (bias && n + e < N) r[e] = r[e] + bias[n + e];
            if (do_scale) r[e] = r[e] * scale;
        }
        if (n + 3 < N && (ldy & 3) == 0) {
            f32x4 v = {r[0], r[1], r[2], r[3]};
            if (rs) { const f32x4 r4 = *reinterpret_cast<const f32x4 *>(rs); v.x = r4.x + v.x; v.y = r4.y + v.y; v.z = r4.z + v.z; v.w = r4.w + v.w; }
            *reinterpret_cast<f32x4 *>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) if (n + e < N) dst[e] = rs ? rs[e] + r[e] : r[e];
        }
    }
}

__global__ void f32_to_f16_kernel(const float *__restrict__ x, _Float16 *__restrict__ y, size_t n4) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n4) return;
    const f32x4 v = reinterpret_cast<const f32x4 *>(x)[i];
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    const f16x4 h = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    reinterpret_cast<f16x4 *>(y)[i] = h;
}
}  // namespace

hipError_t launch_f32_to_f16(const float *x, void *y, size_t n, hipStream_t st) {
    if (n % 4) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f32_to_f16_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, x, reinterpret_cast<_Float16 *>(y), n / 4);
    return hipGetLastError();
}

template <bool XH>
static hipError_t launch_mmf16_t(const uint8_t *W, int n_rows, int K, const void *x, int T, float *y, int ld_out, const float *resid, const float *bias, float scale,
                                 bool do_scale, hipStream_t st) {
    const dim3 big((unsigned)((n_rows + 127) / 128), (unsigned)((T + 127) / 128));
    const char *sw = getenv("MI355_MMF16_TILE");                // "128": always the large tile (A/B and tests)
    if (big.x * big.y >= 256 || (sw && atoi(sw) == 128))
        hipLaunchKernelGGL((mmf16_kernel<2, XH>), big, dim3(256), 0, st, reinterpret_cast<const _Float16 *>(W), n_rows, K, x, T, y, ld_out, resid, bias, scale, (int)do_scale);
    else {
        const dim3 small((unsigned)((n_rows + 63) / 64), (unsigned)((T + 63) / 64));
        hipLaunchKernelGGL((mmf16_kernel<1, XH>), small, dim3(256), 0, st, reinterpret_cast<const _Float16 *>(W), n_rows, K, x, T, y, ld_out, resid, bias, scale, (int)do_scale);
    }
    return hipGetLastError();
}
hipError_t launch_mmf16(const uint8_t *W, int n_rows, int K, const float *x, int T, float *y, int ld_out, const float *resid, hipStream_t st) {
    return launch_mmf16_t<false>(W, n_rows, K, x, T, y, ld_out, resid, nullptr, 1.0f, false, st);
}
// the same product with the activation rows already rounded to f16 (launch_f32_to_f16): [T][K] halves; y = resid + (W x + bias) * scale, every part optional
hipError_t launch_mmf16_xh(const uint8_t *W, int n_rows, int K, const void *xh, int T, float *y, int ld_out, const float *resid, const float *bias, float scale, bool do_scale,
                           hipStream_t st) {
    const char *sw = getenv("MI355_MMF16_LDS");                 // "0": the direct-from-global kernel (A/B and tests)
    if (!(sw && atoi(sw) == 0) && (K % 8) == 0) {
        hipLaunchKernelGGL(mmf16_lds_kernel, dim3((unsigned)((n_rows + 63) / 64), (unsigned)((T + 63) / 64)), dim3(256), 0, st, reinterpret_cast<const _Float16 *>(W), n_rows, K,
                           reinterpret_cast<const _Float16 *>(xh), T, y, ld_out, resid, bias, scale, (int)do_scale);
        return hipGetLastError();
    }
    return launch_mmf16_t<true>(W, n_rows, K, xh, T, y, ld_out, resid, bias, scale, do_scale, st);
}

namespace {
// The encoder's projections (T tokens of one text against f16 weights of a few hundred to a few thousand columns): a product is 19 MB of weights at the most and
// some microseconds of anything, so what counts is one trip to memory, enough workgroups and no launches around it.  Measured on nomic-embed (768 / 3072 columns)
// at 187 tokens, us: 768 x 768 30 with the 64 x 64 direct
// kernel above (36 workgroups, one load in flight, 32 lines per request), gate and up 21 each, down about 60; here, in a pass, output 5.0 and down 8.1, Q | K | V 7.7 and gate | up 10.7, and
// the latter two, of 768 columns, as mmf16_rows_kernel below has them 5.7 and 10.0:
//   * 32 rows x 32 TT tokens per workgroup (144 workgroups for the output at 187 tokens); the NW waves share K, chunk by chunk of 64, and a wave's first PD chunks of
//     both operands - all of them for 768 columns - are requested before the first matrix step;
//   * a request is whole 128-byte lines of eight rows; the operands (16 bytes of 32 rows) are made through LDS of the wave's own, pieces of a row turned by its number.  Asked for as
//     operands, 32 lines per request: gate | up 20.8 us at 187 tokens and 92 at 1800;
//   * partial tiles meet in LDS (rows padded to 36 floats: conflict-free both ways) and are summed in wave order;
//   * two products of the same tokens share a workgroup (NP = 2): gate and up, which leave silu(gate) * up as f16, or the two halves of a head's 64 dimensions of
//     Q | K | V, whose pairs (d, d + 32) are turned by their angle on the way out - Q to its rows, K and V straight into their cells of the f16 cache;
//   * bias and residual are added on the way out.
// XF: the activations are f32 rows, rounded to f16 in registers (the attention's output).
enum { FEW_PLAIN, FEW_SWIGLU, FEW_ROPE };
struct MMF16Few {
    const _Float16 *W, *W2; const void *X;
    float *out; _Float16 *out_h;
    const float *resid, *bias;
    int N, K, T;
    const float *cs; const int32_t *cell; uint16_t *kc, *vc; int n_ctx;       // FEW_ROPE: cos, sin of every token's 32 pairs, the tokens' cells, the layer's cache planes
};
template <int NW, int EPI, int TT, int PD, bool XF>
__global__ __launch_bounds__(64 * NW, EPI == FEW_SWIGLU && NW == 4 && TT == 1 ? 3 : 1) void mmf16_few_kernel(const MMF16Few a) {
    constexpr int NP = EPI == FEW_PLAIN ? 1 : 2, ROWS = EPI == FEW_ROPE ? 64 : 32;
    constexpr int LD = 36, LDR = 64, STAGE = (NP + TT) * 32 * LDR;                                     // floats per row of a partial tile; halves per row of a staged chunk
    constexpr int PART_BYTES = NW * NP * TT * 32 * LD * 4, STAGE_BYTES = NW * STAGE * 2;
    __shared__ __attribute__((aligned(16))) uint8_t smem[PART_BYTES > STAGE_BYTES ? PART_BYTES : STAGE_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), m = lane & 31, kg = lane >> 5;
    const int n0 = blockIdx.x * ROWS, t0 = blockIdx.y * (32 * TT), r8 = lane >> 3, c8 = 8 * (lane & 7);
    float *part = reinterpret_cast<float *>(smem);
    _Float16 *stage = reinterpret_cast<_Float16 *>(smem) + wave * STAGE;
    // request i of an operand tile: row r8 + 8 i, its halves c8 .. of the chunk; rows past the end read the last one (their results are never stored)
    unsigned wrow[4], xrow[TT][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int g = n0 + r8 + 8 * i;
        wrow[i] = (unsigned)(g < a.N ? g : a.N - 1) * (unsigned)a.K + c8;
#pragma unroll
        for (int t = 0; t < TT; t++) { const int h = t0 + 32 * t + r8 + 8 * i; xrow[t][i] = (unsigned)(h < a.T ? h : a.T - 1) * (unsigned)a.K + c8; }
    }
    const _Float16 *W[NP] = {a.W};
    if constexpr (NP == 2) W[1] = a.W2;
    struct Slot { f16x8 w[NP][4]; f16x8 x[TT][XF ? 1 : 4]; f32x4 xf[TT][XF ? 8 : 1]; };
    Slot s[PD];
    const int nc = a.K >> 6, cn = wave < nc ? (nc - wave + NW - 1) / NW : 0;                          // this wave's chunks: wave, wave + NW, ..
    const int last = nc - 1;
    auto fetch = [&](Slot &v, int i) {
        const unsigned k = 64u * (unsigned)(wave + NW * i < last ? wave + NW * i : last);
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int p = 0; p < NP; p++) v.w[p][j] = *reinterpret_cast<const f16x8 *>(W[p] + (wrow[j] + k));
#pragma unroll
            for (int t = 0; t < TT; t++) {
                if constexpr (XF) {
                    const float *x = reinterpret_cast<const float *>(a.X) + (xrow[t][j] + k);
                    v.xf[t][2 * j] = *reinterpret_cast<const f32x4 *>(x); v.xf[t][2 * j + 1] = *reinterpret_cast<const f32x4 *>(x + 4);
                } else v.x[t][j] = *reinterpret_cast<const f16x8 *>(reinterpret_cast<const _Float16 *>(a.X) + (xrow[t][j] + k));
            }
        }
    };
    f32x16 acc[NP][TT];
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[p][t][r] = 0.0f;
    auto put = [&](const Slot &v) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            _Float16 *d = stage + (r8 + 8 * j) * LDR + (c8 ^ (8 * r8));          // (piece c of row r at c ^ (r & 7): no bank conflicts, and no padding)
#pragma unroll
            for (int p = 0; p < NP; p++) *reinterpret_cast<f16x8 *>(d + p * 32 * LDR) = v.w[p][j];
#pragma unroll
            for (int t = 0; t < TT; t++) {
                f16x8 b;
                if constexpr (XF) {
#pragma unroll
                    for (int e = 0; e < 4; e++) { b[e] = (_Float16)v.xf[t][2 * j][e]; b[4 + e] = (_Float16)v.xf[t][2 * j + 1][e]; }
                } else b = v.x[t][j];
                *reinterpret_cast<f16x8 *>(d + (NP + t) * 32 * LDR) = b;
            }
        }
    };
    auto use = [&]() {
        const _Float16 *f = stage + m * LDR;
        const int x = 8 * (m & 7);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            f16x8 w[NP];
#pragma unroll
            for (int p = 0; p < NP; p++) w[p] = *reinterpret_cast<const f16x8 *>(f + p * 32 * LDR + ((16 * j + 8 * kg) ^ x));
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const f16x8 b = *reinterpret_cast<const f16x8 *>(f + (NP + t) * 32 * LDR + ((16 * j + 8 * kg) ^ x));
#pragma unroll
                for (int p = 0; p < NP; p++) acc[p][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[p], b, acc[p][t], 0, 0, 0);
            }
        }
    };
#pragma unroll
    for (int u = 0; u < PD; u++) { fetch(s[u], u); __builtin_amdgcn_sched_barrier(0); }               // (in the order of their use: a wait for one slot is not one for the next)
    // what a plain product adds on its way out, behind them (asked for there it was a trip to memory of its own, 0.3 to 0.5 us a launch): a thread's outputs are all of one weight row
    constexpr int NE = (1024 * TT + 64 * NW - 1) / (64 * NW);
    const int er = tid & 31, en = n0 + er;
    float rv[EPI == FEW_PLAIN ? NE : 1], bv = 0.0f;
    if constexpr (EPI == FEW_PLAIN) {
        const int nn = en < a.N ? en : a.N - 1;
        if (a.bias) bv = a.bias[nn];
        if (a.resid) {
#pragma unroll
            for (int j = 0; j < NE; j++) { const int g = t0 + (tid >> 5) + 2 * NW * j; rv[j] = a.resid[(size_t)(g < a.T ? g : a.T - 1) * a.N + nn]; }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    int i = 0;
    for (; i + PD < cn; i += PD)                             // (no branch around a request: it would become a wait for all of them)
#pragma unroll
        for (int u = 0; u < PD; u++) {
            put(s[u]);
            __builtin_amdgcn_sched_barrier(0);               // (a wave's LDS accesses are made in order)
            fetch(s[u], i + PD + u);
            __builtin_amdgcn_sched_barrier(0);
            use();
        }
#pragma unroll
    for (int u = 0; u < PD; u++) if (i + u < cn) { put(s[u]); __builtin_amdgcn_wave_barrier(); use(); __builtin_amdgcn_wave_barrier(); }
    __syncthreads();                                         // the partial tiles take the staging area's place
    // register r of a lane: weight row (r & 3) + 8 (r >> 2) + 4 kg, token = lane & 31
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<f32x4 *>(part + (((wave * NP + p) * TT + t) * 32 + m) * LD + 8 * q + 4 * kg) =
                    f32x4{acc[p][t][4 * q], acc[p][t][4 * q + 1], acc[p][t][4 * q + 2], acc[p][t][4 * q + 3]};
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int row = er, t = (tid >> 5) + 2 * NW * j, gt = t0 + t, n = en;
        if (t >= 32 * TT) break;
        float v[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            v[p] = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; w++) v[p] += part[(((w * NP + p) * TT + (t >> 5)) * 32 + (t & 31)) * LD + row];
        }
        if (gt >= a.T || n >= a.N) continue;
        if constexpr (EPI == FEW_ROPE) {
            const int E = a.N / 3, s = n0 / E, c0 = n0 - s * E;         // (a head is a whole tile, a segment whole heads)
            float y0 = v[0], y1 = v[1];
            if (s < 2) {
                const float c = a.cs[(size_t)gt * 64 + 2 * row], sn = a.cs[(size_t)gt * 64 + 2 * row + 1];
                y0 = v[0] * c - v[1] * sn;
                y1 = v[0] * sn + v[1] * c;
            }
            if (s == 0) { float *q = a.out + (size_t)gt * E + c0 + row; q[0] = y0; q[32] = y1; }
            else { uint16_t *d = (s == 1 ? a.kc : a.vc) + ((size_t)(c0 >> 6) * a.n_ctx + a.cell[gt]) * 64 + row; d[0] = f2h(y0); d[32] = f2h(y1); }
        } else {
            const size_t o = (size_t)gt * a.N + n;
            if constexpr (EPI == FEW_SWIGLU) a.out_h[o] = (_Float16)((v[0] / (1.0f + expf(-v[0]))) * v[1]);
            else {
                float y = v[0];
                if (a.bias) y = y + bv;
                if (a.resid) y = rv[j] + y;
                a.out[o] = y;
            }
        }
    }
}
// Two products of the same tokens (gate and up, or the halves of 64-wide heads) where K is at most ROWS_K columns and there are few workgroups: 32 rows of each x 32 tokens per workgroup, whose
// activation rows are whole in LDS, staged once by all; of the eight waves four take the one product and four the other, a chunk of 64 columns in four each, all of a wave's weights
// requested at once.  What bounds such a launch is a wave's own chain of instructions - one or two waves a SIMD, some thousand of them - and in the form above a wave stages both products and the
// tokens for itself (both forms' times: few_two).  Twelve waves, two chunks each: no faster and, with one workgroup a CU, gate | up of 187 tokens 11.8 instead of 9.1 us.  With the LayerNorm in front
// of it in the launch, every workgroup norming its rows: 7.9 and 15.1 instead of 5.1 and 9.1, a launch of the norm is 2.7.  (These back to back, half a microsecond to one less than in a pass.)
constexpr int ROWS_K = 768;
template <int EPI>
__global__ __launch_bounds__(512, 4) void mmf16_rows_kernel(const MMF16Few a) {
    constexpr int ROWS = EPI == FEW_ROPE ? 64 : 32, KJ = ROWS_K / 64, NK = 4, PD = KJ / NK, LD = 36;
    constexpr int X_BYTES = 32 * KJ * 128, W_BYTES = 8 * 4096;
    static_assert(8 * 32 * LD * 4 <= X_BYTES + W_BYTES && KJ % NK == 0 && KJ % 2 == 0, "the partial tiles take the operands' place");
    __shared__ __attribute__((aligned(16))) uint8_t smem[X_BYTES + W_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), p = wave & 1, ks = wave >> 1, m = lane & 31, kg = lane >> 5;
    const int n0 = blockIdx.x * ROWS, t0 = blockIdx.y * 32, nc = a.K >> 6, r8 = lane >> 3, c8 = lane & 7;
    uint8_t *const sx = smem, *const sw = smem + X_BYTES + wave * 4096;
    // the tokens' rows, sixteen threads a row (past the end the last one's; a piece past K is the thread's first, and not staged: K is 128 or more), then the wave's chunks of its product's rows
    const int row = tid >> 4, l16 = tid & 15;
    f16x8 v[KJ / 2];
    {
        const int gt = t0 + row < a.T ? t0 + row : a.T - 1;
        const unsigned o = ((unsigned)gt * (unsigned)a.K + 8u * l16) * 2u;
#pragma unroll
        for (int j = 0; j < KJ / 2; j++) v[j] = *reinterpret_cast<const f16x8 *>(reinterpret_cast<const uint8_t *>(a.X) + (o + (128 * j + 8 * l16 < a.K ? 256u * j : 0u)));
    }
    __builtin_amdgcn_sched_barrier(0);
    const uint8_t *const W = reinterpret_cast<const uint8_t *>(p ? a.W2 : a.W);
    unsigned wrow[4];
#pragma unroll
    for (int i = 0; i < 4; i++) { const int g = n0 + r8 + 8 * i; wrow[i] = ((unsigned)(g < a.N ? g : a.N - 1) * (unsigned)a.K + 8u * c8) * 2u; }
    f16x8 w[PD][4];
#pragma unroll
    for (int u = 0; u < PD; u++) {
        const unsigned k = 128u * (unsigned)(ks + NK * u < nc ? ks + NK * u : nc - 1);
#pragma unroll
        for (int j = 0; j < 4; j++) w[u][j] = *reinterpret_cast<const f16x8 *>(W + (wrow[j] + k));
        __builtin_amdgcn_sched_barrier(0);
    }
    // a thread's output: a token and a pair of rows of either product; what the pairs are turned by, and their cell
    const int et = tid >> 4, er = 2 * (tid & 15), gt = t0 + et;
    f32x4 cv = {0.0f, 0.0f, 0.0f, 0.0f};
    int cl = 0;
    if constexpr (EPI == FEW_ROPE) { const int q = gt < a.T ? gt : a.T - 1; cv = *reinterpret_cast<const f32x4 *>(a.cs + (size_t)q * 64 + 2 * er); cl = a.cell[q]; }
    __builtin_amdgcn_sched_barrier(0);
    // (a chunk of a row is 128 bytes; piece c of row r at c ^ (r & 7): no bank conflicts either way)
#pragma unroll
    for (int j = 0; j < KJ / 2; j++) { const int c = 2 * j + (l16 >> 3); if (c < nc) *reinterpret_cast<f16x8 *>(sx + (row * KJ + c) * 128 + 16 * ((l16 & 7) ^ (row & 7))) = v[j]; }
    __syncthreads();
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
    for (int u = 0; u < PD; u++) {
        const int c = ks + NK * u;
        if (c < nc) {
#pragma unroll
            for (int j = 0; j < 4; j++) *reinterpret_cast<f16x8 *>(sw + (r8 + 8 * j) * 128 + 16 * (c8 ^ r8)) = w[u][j];
            __builtin_amdgcn_wave_barrier();                 // (a wave's LDS accesses are made in order)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int o = 16 * ((2 * j + kg) ^ (m & 7));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8 *>(sw + m * 128 + o), *reinterpret_cast<const f16x8 *>(sx + (m * KJ + c) * 128 + o), acc, 0, 0, 0);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    float *const part = reinterpret_cast<float *>(smem);     // (registers as in mmf16_few_kernel)
#pragma unroll
    for (int q = 0; q < 4; q++) *reinterpret_cast<f32x4 *>(part + (wave * 32 + m) * LD + 8 * q + 4 * kg) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    if (gt >= a.T || n0 + er >= a.N) return;
    f32x2 y[2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
#pragma unroll
    for (int k = 0; k < NK; k++)
#pragma unroll
        for (int q = 0; q < 2; q++) y[q] += *reinterpret_cast<const f32x2 *>(part + ((2 * k + q) * 32 + et) * LD + er);
    if constexpr (EPI == FEW_SWIGLU) {
        *reinterpret_cast<f16x2 *>(a.out_h + (size_t)gt * a.N + n0 + er) = f16x2{(_Float16)((y[0].x / (1.0f + expf(-y[0].x))) * y[1].x), (_Float16)((y[0].y / (1.0f + expf(-y[0].y))) * y[1].y)};
    } else {
        const int E = a.N / 3, s = (n0 >= E) + (n0 >= 2 * E), c0 = n0 - s * E;         // (a head is a whole tile, a segment whole heads)
        if (s < 2) {
            const f32x2 c = {cv.x, cv.z}, sn = {cv.y, cv.w}, b0 = y[0], b1 = y[1];
            y[0] = b0 * c - b1 * sn;
            y[1] = b0 * sn + b1 * c;
        }
        if (s == 0) { float *q = a.out + (size_t)gt * E + c0 + er; *reinterpret_cast<f32x2 *>(q) = y[0]; *reinterpret_cast<f32x2 *>(q + 32) = y[1]; }
        else {
            uint16_t *d = (s == 1 ? a.kc : a.vc) + ((size_t)(c0 >> 6) * a.n_ctx + cl) * 64 + er;
            *reinterpret_cast<unsigned *>(d) = (unsigned)f2h(y[0].x) | ((unsigned)f2h(y[0].y) << 16);
            *reinterpret_cast<unsigned *>(d + 32) = (unsigned)f2h(y[1].x) | ((unsigned)f2h(y[1].y) << 16);
        }
    }
}
template <int NW, int EPI, int TT, int PD, bool XF>
void few_go(const MMF16Few &a, hipStream_t st) {
    const int rows = EPI == FEW_ROPE ? 64 : 32;
    hipLaunchKernelGGL((mmf16_few_kernel<NW, EPI, TT, PD, XF>), dim3((unsigned)((a.N + rows - 1) / rows), (unsigned)((a.T + 32 * TT - 1) / (32 * TT))), dim3(64 * NW), 0, st, a);
}
// two products: the form above, or a workgroup's waves sharing K.  Of the latter two token tiles per workgroup, the weights read half as often, once there are enough workgroups
template <int NW, int EPI>
void few_two(const MMF16Few &a, hipStream_t st) {
    const int rows = EPI == FEW_ROPE ? 64 : 32, wg = (a.N + rows - 1) / rows * ((a.T + 31) / 32);
    // us in a pass of 768 columns, that form / the shared K, medians of two profiled runs of each in turn, at 40, 187, 300, 400, 500, 600, 700, 800, 900, 1000, 1400, 1800 and 2000 tokens:
    //   Q | K | V   5.4 / 7.0, 5.7 / 7.7, 7.3 / 8.8, 7.6 / 9.3, 9.5 / 11.8, 10.1 / 14.1, 11.3 / 13.8, 11.8 / 14.3, 13.4 / 15.9, 14.1 / 18.6, 18.2 / 22.7, 21.8 / 25.7, 23.3 / 29.4
    //   gate | up   6.0 / 6.1, 10.1 / 10.7, 12.3 / 12.7, 14.8 / 15.1, 17.0 / 17.0, 20.5 / 20.4, 22.5 / 23.4, 24.8 / 24.2, 27.1 / 27.4, 29.2 / 27.7, 39.2 / 37.4, 49.3 / 45.2, 54.1 / 49.1
    // So Q | K | V at any number, gate | up to nine workgroups a CU (768 tokens of 3072 rows)
    if (a.K >= 128 && a.K <= ROWS_K && a.N % 32 == 0 && (EPI == FEW_ROPE || wg <= 9 * num_cu())) {
        hipLaunchKernelGGL((mmf16_rows_kernel<EPI>), dim3((unsigned)(a.N / rows), (unsigned)((a.T + 31) / 32)), dim3(512), 0, st, a);
        return;
    }
    if (wg * (rows / 32) >= 1280) few_go<NW, EPI, 2, 2, false>(a, st);
    else few_go<NW, EPI, 1, EPI == FEW_SWIGLU && NW == 4 ? 2 : 3, false>(a, st);
}
// A plain product, us back to back, K 768 of f32 rows / K 3072 of halves, both to 768 rows.  What counts is a wave's own chain again, so as many waves as K gives chunks where a CU has one workgroup: 187 tokens,
// twelve waves 3.8 / 7.1, four and eight 4.3 / 7.5.  Beyond, in rounds of a workgroup a CU: f32 rows on four waves (400 tokens 6.0, twelve 6.4; 1000 8.3, 10.2); halves on one, two or three token
// tiles, whose rounds take about 7.1, 9.4 and 14.6: 400 tokens 12.5, 9.3, 12.6, 800 about 18.5, 18.4, 14.8, 1200 24.8, 19.2, 27.0, 2048 36.9, 29.5, 38.9; eight waves with one and, from 1280
// workgroups on, two 13.2, 19.9, 26.6, 31.1.
template <bool XF>
void few_plain(const MMF16Few &a, hipStream_t st) {
    const int cu = num_cu(), gx = (a.N + 31) / 32, gy = (a.T + 31) / 32;
    if constexpr (XF) {
        if (a.K > 1024) few_go<8, FEW_PLAIN, 1, 2, true>(a, st);
        else if (gx * gy <= cu) few_go<12, FEW_PLAIN, 1, 1, true>(a, st);
        else few_go<4, FEW_PLAIN, 1, 2, true>(a, st);
        return;
    } else {
        if (a.K <= 1024) {
            if (gx * gy >= 1280) few_go<4, FEW_PLAIN, 2, 2, false>(a, st); else few_go<4, FEW_PLAIN, 1, 3, false>(a, st);
            return;
        }
        const auto time = [&](int tt, int round) { return (gx * ((gy + tt - 1) / tt) + cu - 1) / cu * round; };
        const int one = time(1, 71), two = time(2, 94), three = time(3, 146);
        if (one <= two && one <= three) few_go<12, FEW_PLAIN, 1, 2, false>(a, st);
        else if (two <= three) few_go<12, FEW_PLAIN, 2, 1, false>(a, st);
        else few_go<8, FEW_PLAIN, 3, 2, false>(a, st);
    }
}
}  // namespace

bool mmf16_few_applicable(int n_rows, int K, int T) {
    return T >= 8 && n_rows >= 32 && K % 64 == 0 && (size_t)n_rows * K < (1ull << 31) && (size_t)T * K < (1ull << 31);
}
// out[t][n_rows] = W X (+ bias) (+ resid); X: [T][K] halves (x_f16) or floats, rounded to f16
hipError_t launch_mmf16_few(const uint8_t *W, int n_rows, int K, const void *x, bool x_f16, int T, float *out, const float *resid, const float *bias, hipStream_t st) {
    MMF16Few a{};
    a.W = reinterpret_cast<const _Float16 *>(W); a.X = x; a.N = n_rows; a.K = K; a.T = T; a.out = out; a.resid = resid; a.bias = bias;
    if (x_f16) few_plain<false>(a, st); else few_plain<true>(a, st);
    return hipGetLastError();
}
// out[t][n_rows] = f16(silu(W_gate x) * (W_up x)), x: [T][K] halves
hipError_t launch_mmf16_few_swiglu(const uint8_t *W_gate, const uint8_t *W_up, int n_rows, int K, const void *xh, int T, void *out_h, hipStream_t st) {
    MMF16Few a{};
    a.W = reinterpret_cast<const _Float16 *>(W_gate); a.W2 = reinterpret_cast<const _Float16 *>(W_up); a.X = xh; a.N = n_rows; a.K = K; a.T = T;
    a.out_h = reinterpret_cast<_Float16 *>(out_h);
    if (K > 1024) few_two<8, FEW_SWIGLU>(a, st); else few_two<4, FEW_SWIGLU>(a, st);
    return hipGetLastError();
}
// the projections of E = n_head * 64 rows each of W (Q | K | V) for x: [T][K] halves; rope pairs (d, d + 32) by cs[T][64]; q [T][E], k and v into the f16 cache
hipError_t launch_mmf16_few_qkv_rope(const uint8_t *W, int E, int K, const void *xh, int T, float *q, const float *cs, const int32_t *cell, KVLayerView kv, int n_ctx, hipStream_t st) {
    if (E % 64) return hipErrorInvalidValue;
    MMF16Few a{};
    a.W = reinterpret_cast<const _Float16 *>(W); a.W2 = a.W + (size_t)32 * K; a.X = xh; a.N = 3 * E; a.K = K; a.T = T;
    a.out = q; a.cs = cs; a.cell = cell; a.kc = reinterpret_cast<uint16_t *>(kv.k); a.vc = reinterpret_cast<uint16_t *>(kv.v); a.n_ctx = n_ctx;
    if (K > 1024) few_two<8, FEW_ROPE>(a, st); else few_two<4, FEW_ROPE>(a, st);
    return hipGetLastError();
}

}  // namespace mi355
