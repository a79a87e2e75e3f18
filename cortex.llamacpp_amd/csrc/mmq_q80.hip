// mmq_q80.hip — prompt batches against Q8_0 weights on the matrix cores (mul_mat_q for Q8_0).
//
//   out[t][r] = sum over 32-blocks b of  (float)isum_b * (d_w[r][b] * d_a[t][b]),   isum_b = sum_{k in b} w[r][k] * a[t][k]
//
// exactly ggml_vec_dot_q8_0_q8_0: integer block sums, one f32 multiply-add per block, blocks added in order — so unlike
// the K-quant kernels (whose super-block sums are re-associated) this one reproduces the CPU result bit for bit.
//
// An MFMA contracts K = 32 = one Q8_0 block (v_mfma_i32_32x32x32_i8 or 16x16x32): A = tokens x 32 codes, B = weight rows x
// 32 codes, so the result tile holds some tokens of one weight row per lane.
#include "kernels.h"
#include "quant_dev.h"

namespace mi355 {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// up to three tensors of K columns that share the activations, one launch: tensor i is the workgroups from tile0[i] on
struct Q80Args {
    const uint8_t *W[3]; size_t row_bytes;
    float *out[3];
    int n_rows[3], ld_out[3], tile0[3];
    int n_seg, K, T;
    const int8_t *aq; const uint16_t *ad; const float *resid;
};

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
template <int SZ> struct Tile;
template <> struct Tile<32> {
    using Codes = i32x4; using Ints = i32x16; using Floats = f32x16;
    __device__ static Ints dot(const Codes &x, const Codes &w, const Ints &z) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w, z, 0, 0, 0); }
    __device__ static Floats outer(f16x4 x, f16x4 w, const Floats &z) { return __builtin_amdgcn_mfma_f32_32x32x8f16(x, w, z, 0, 0, 0); }
};
template <> struct Tile<16> {
    using Codes = long; using Ints = i32x4; using Floats = f32x4;
    __device__ static Ints dot(const Codes &x, const Codes &w, const Ints &z) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(x, w, z, 0, 0, 0); }
    __device__ static Floats outer(f16x4 x, f16x4 w, const Floats &z) { return __builtin_amdgcn_mfma_f32_16x16x16f16(x, w, z, 0, 0, 0); }
};

// Rows come in steps of U blocks, 128 or 256 bytes.  A lane that reads its own row from memory costs the CU's address unit a clock a lane, and in the matrix unit's layout every lane is another
// line: a row of 64 blocks took 20 us however few the tiles (2048 x 2048, 40 tokens; its products are 5).  So a wave instruction brings eight (four) rows' steps into LDS - S of them in
// turn, the 16-byte pieces of row i in the order p ^ (i & 7), so that the matrix unit's reads meet no bank twice -, and the four waves share both operands.  The scales come the same way, and
// their products from the matrix unit too: one f16 contraction of which all elements but one are zero IS d_w * d_a of every output, exactly (22 bits in f32, subnormals kept), in place of a
// vector instruction a result.  What is left to the vector unit is convert (or subtract), multiply, add - the CPU's three roundings an output and block in the CPU's order -: 48 instructions a 32 x 32
// tile and block, its bound (5632 x 2048, 2000 tokens: 63 us of 97).
// Wave = W x W tiles of SZ x SZ, workgroup = 2 x 2 waves.  Tiles of 16 take steps of eight blocks: what they wait for is a barrier and two LDS reads a step (four / eight, 40 tokens:
// 2048 x 2048 7.3 / 6.5, 2048 x 5632 16.8 / 14.6, 4096 x 14336 41 / 35; tiles of 32 the same either way).
// us, 40 / 611 / 2000 tokens, this | every lane its own row, scales from LDS: 2048 x 2048 6.5 / 17 / 39 | 21 / 35 / 61, 5632 x 2048 9.6 / 35 / 97 | 22 / 60 / 151, 4096 x 14336
// 35 / 152 / 415 | 133 / 349 / 582, 1024 x 4096 10.6 / 22 / 37 | 38 / 38 / 69.
// (Tried: rows straight from memory in tiles of 16, or two to four steps ahead: the same 20 us.  The products of the next tile asked for before the fold of this one: nothing.)
template <int SZ, int W, int S, int U>
__global__ __launch_bounds__(256, 2) void mmq_q80_tiles_kernel(const Q80Args a) {
    using TL = Tile<SZ>;
    using Codes = typename TL::Codes;
    // rows of either operand, 32 U B of codes and 2 U of scales each; a scale request brings SQ rows'
    constexpr int ROWS = 2 * SZ * W, RB = 32 * U, PIECES = 2 * U, STEP = 2 * RB * ROWS, SB = 2 * U, SQ = U == 4 ? 32 : 64, SOP = (ROWS + SQ - 1) / SQ * SQ * SB, STAGE = STEP + 2 * SOP;
    constexpr int NR = SZ * SZ / 64, NC = ROWS * RB / 4096, SR = (ROWS + SQ - 1) / SQ, NS = SR > 2 ? SR / 2 : 1, LOADS = 2 * NC + NS;
    __shared__ __attribute__((aligned(1024))) uint8_t sm[S * STAGE];
    int sg = 0;
    if (a.n_seg > 1 && (int)blockIdx.x >= a.tile0[1]) sg = 1;
    if (a.n_seg > 2 && (int)blockIdx.x >= a.tile0[2]) sg = 2;
    const int n_rows = a.n_rows[sg], K = a.K, T = a.T, nb = K >> 5, steps = nb / U;
    const int l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), n = l & (SZ - 1), kg = l / SZ;
    const int t0 = blockIdx.y * ROWS, r0 = ((int)blockIdx.x - a.tile0[sg]) * ROWS;
    const int last_r = (n_rows - r0 < ROWS ? n_rows - r0 : ROWS) - 1, last_t = (T - t0 < ROWS ? T - t0 : ROWS) - 1;
    const uint8_t *const wbase = (const uint8_t *)uniform_ptr(a.W[sg] + (size_t)r0 * a.row_bytes);
    const uint8_t *const xbase = (const uint8_t *)uniform_ptr(a.aq + (size_t)t0 * K), *const dbase = (const uint8_t *)uniform_ptr(a.ad + (size_t)t0 * nb);
    // a request: 1 KB of codes, the 16-byte pieces of row i in the order p ^ (i & 7); or SQ rows' scales
    unsigned woff[NC], xoff[NC], soff[NS];
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int r = (wave + 4 * i) * (1024 / RB) + l / PIECES;
        const unsigned piece = 16u * ((l % PIECES) ^ (r & 7));
        woff[i] = (unsigned)(r < last_r ? r : last_r) * (unsigned)a.row_bytes + piece;
        xoff[i] = (unsigned)(r < last_t ? r : last_t) * (unsigned)K + piece;
    }
    bool sw[NS];
    unsigned sto[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const int q = (wave + 4 * i) % (2 * SR), r = (q % SR) * SQ + (U == 4 ? l >> 1 : l);
        const unsigned half = U == 4 ? 4u * (l & 1) : 0u;
        sw[i] = q < SR;
        sto[i] = STEP + q * (SQ * SB);
        soff[i] = sw[i] ? (unsigned)(r < last_r ? r : last_r) * (unsigned)a.row_bytes + (unsigned)K + half : (unsigned)(r < last_t ? r : last_t) * (unsigned)nb * 2u + half;
    }
    const unsigned lds = __builtin_amdgcn_readfirstlane((int)(unsigned)(uintptr_t)sm);
    const auto ask = [&](int step, int buf) {
        const int s = step < steps ? step : steps - 1;                 // (past the end: the last again, never read)
        const unsigned to = lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < NC; i++) lds_dma16(wbase + (size_t)s * RB, woff[i], to + (wave + 4 * i) * 1024);
#pragma unroll
        for (int i = 0; i < NC; i++) lds_dma16(xbase + (size_t)s * RB, xoff[i], to + STEP / 2 + (wave + 4 * i) * 1024);
#pragma unroll
        for (int i = 0; i < NS; i++) {
            if constexpr (U == 4) lds_dma4((sw[i] ? wbase : dbase) + (size_t)s * SB, soff[i], to + sto[i]);
            else lds_dma16((sw[i] ? wbase : dbase) + (size_t)s * SB, soff[i], to + sto[i]);
        }
    };
    const int wr = (wave & 1) * SZ * W, wt = (wave >> 1) * SZ * W;     // the wave's tiles in the workgroup's
    const uint32_t first = kg == 0 ? 0x0000ffffu : 0u, second = kg == 0 ? 0xffff0000u : 0u;
    const auto one = [&](const auto &d, int u) { return __builtin_bit_cast(f16x4, u32x2{d[u >> 1] & ((u & 1) ? second : first), 0u}); };
    float acc[W][W][NR];
#pragma unroll
    for (int i = 0; i < W; i++)
#pragma unroll
        for (int j = 0; j < W; j++)
#pragma unroll
            for (int r = 0; r < NR; r++) acc[i][j][r] = 0.0f;
    // (with the bias as the sums' start a subtraction converts them: 4096 x 14336 at 40 tokens, tiles of 16 in steps of four blocks, 44 -> 41 us, at 2000, four of 32 a wave, 430 -> 415; one of 32 a wave is 4 % slower for it)
    constexpr bool BIAS = SZ == 16 || W == 2;
    const typename TL::Ints zi = (typename TL::Ints)(BIAS ? INT_BIAS : 0);
    const typename TL::Floats zf = {};
#pragma unroll
    for (int s = 0; s + 1 < S; s++) ask(s, s);
    int buf = 0;
    for (int step = 0; step < steps; step++) {
        asm volatile("s_waitcnt vmcnt(%c0) lgkmcnt(0)\n\ts_barrier" :: "i"(LOADS * (S - 2)) : "memory");
        ask(step + S - 1, buf ? buf - 1 : S - 1);
        const uint8_t *const at = sm + buf * STAGE;
        buf = buf + 1 < S ? buf + 1 : 0;
        typedef unsigned int scales __attribute__((ext_vector_type(U / 2)));
        scales dw[W], da[W];
#pragma unroll
        for (int i = 0; i < W; i++) {
            dw[i] = *reinterpret_cast<const scales *>(at + STEP + (wr + SZ * i + n) * SB);
            da[i] = *reinterpret_cast<const scales *>(at + STEP + SOP + (wt + SZ * i + n) * SB);
        }
        const auto codes = [&](const uint8_t *op, int row, int u) {
            if constexpr (SZ == 32) return *reinterpret_cast<const Codes *>(op + row * RB + (((2 * u + kg) ^ (n & 7)) * 16));
            else return *reinterpret_cast<const Codes *>(op + row * RB + (((2 * u + (kg >> 1)) ^ (n & 7)) * 16) + (kg & 1) * 8);
        };
        Codes w[2][W], x[2][W];
        const auto read = [&](int u) {
#pragma unroll
            for (int i = 0; i < W; i++) { w[u & 1][i] = codes(at, wr + SZ * i + n, u); x[u & 1][i] = codes(at + STEP / 2, wt + SZ * i + n, u); }
        };
        read(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u + 1 < U) read(u + 1);
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < W; j++) {
                    const auto c = TL::dot(x[u & 1][j], w[u & 1][i], zi);
                    const auto sc = TL::outer(one(da[j], u), one(dw[i], u), zf);
#pragma unroll
                    for (int r = 0; r < NR; r++) acc[i][j][r] = acc[i][j][r] + (BIAS ? biased_f32(c[r]) : (float)c[r]) * sc[r];
                }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                   // nothing lands in LDS after the workgroup's end
    const int ld = a.ld_out[sg];
#pragma unroll
    for (int i = 0; i < W; i++) {
        const int row = r0 + wr + SZ * i + n;
        if (row >= n_rows) continue;
        float *const out = a.out[sg] + row;
#pragma unroll
        for (int j = 0; j < W; j++) {
            const auto token = [&](int r) { return t0 + wt + SZ * j + (SZ == 32 ? 8 * (r >> 2) + 4 * kg + (r & 3) : 4 * kg + r); };
            if (a.resid) {                                             // (may be out itself; the tile's are requested before its first is stored)
                float old[NR];
#pragma unroll
                for (int r = 0; r < NR; r++) old[r] = a.resid[(size_t)(token(r) < T ? token(r) : T - 1) * ld + row];
#pragma unroll
                for (int r = 0; r < NR; r++) acc[i][j][r] = old[r] + acc[i][j][r];
            }
#pragma unroll
            for (int r = 0; r < NR; r++)
                if (token(r) < T) out[(size_t)token(r) * ld] = acc[i][j][r];
        }
    }
}

}  // namespace

// Q4_0 / Q5_0 / IQ4_NL rows as Q8_0 device rows ([codes K][scales K/32]): code = nibble - 8, (nibble | fifth bit) - 16, level[nibble] - all int8 -
// with the block's own f16 scale.  The copy is EXACT (same integers, same scales), so the kernel above computes the same block sums as the format's
// own vec_dot; it is made once at load for prompt batches (1.06 B per weight beside the file's 0.56 - 0.69).
__global__ __launch_bounds__(256) void expand_nib32_q80_kernel(int type, const uint8_t *__restrict__ W, size_t row_bytes, int n_rows, int K, uint8_t *__restrict__ dst,
                                                               size_t dst_row) {
    const int row = blockIdx.y;
    const int nblk = K >> 5;
    const size_t half = (size_t)K >> 1;
    const uint8_t *r = W + (size_t)row * row_bytes;
    uint8_t *o = dst + (size_t)row * dst_row;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < K; e += gridDim.x * 256) {
        const int b = e >> 5, j = e & 31;
        const int nib = (r[(size_t)b * 16 + (j & 15)] >> (4 * (j >> 4))) & 0x0f;
        int code;
        if (type == T_Q4_0) code = nib - 8;
        else if (type == T_Q5_0) {
            const uint32_t qh = *reinterpret_cast<const uint32_t *>(r + half + (size_t)b * 4);
            code = (nib | (int)(((qh >> j) & 1u) << 4)) - 16;
        } else code = iq4nl_value(nib);
        o[e] = (uint8_t)(int8_t)code;
        if (j == 0) {
            const uint16_t d = *reinterpret_cast<const uint16_t *>(r + half + (type == T_Q5_0 ? (size_t)nblk * 4 : 0) + (size_t)b * 2);
            *reinterpret_cast<uint16_t *>(o + (size_t)K + (size_t)b * 2) = d;
        }
    }
}
size_t mmq_q80_copy_bytes(int type, int64_t n_rows, int K) {
    if ((type != T_Q4_0 && type != T_Q5_0 && type != T_IQ4_NL) || (K % 32) != 0 || K > 65536) return 0;
    return (size_t)n_rows * dev_row_bytes(T_Q8_0, K);
}
hipError_t launch_expand_q80_copy(int type, const uint8_t *W, size_t row_bytes, int n_rows, int K, uint8_t *dst, hipStream_t st) {
    if (!mmq_q80_copy_bytes(type, n_rows, K)) return hipErrorInvalidValue;
    for (int r0 = 0; r0 < n_rows; r0 += 65535) {
        const int nr = n_rows - r0 < 65535 ? n_rows - r0 : 65535;
        hipLaunchKernelGGL(expand_nib32_q80_kernel, dim3((unsigned)((K + 255) / 256 < 8 ? (K + 255) / 256 : 8), nr), dim3(256), 0, st, type, W + (size_t)r0 * row_bytes, row_bytes, nr, K,
                           dst + (size_t)r0 * dev_row_bytes(T_Q8_0, K), dev_row_bytes(T_Q8_0, K));
    }
    return hipGetLastError();
}

// The mat-vec takes one, two or four tokens to a pass over the weights; from three on they go here (us of a batch, mat-vec | tiles, 3 / 4 / 5 / 16 / 31 tokens: six TinyLlama-1.1B Q8_0 layers
// 533 444 604 1056 2138 | 422 428 426 434 451, four 8B ones 723 671 888 1571 3294 | 583 577 577 590 614, as Q4_0 with the copy above 615 655 - 1651 3327 | 571 569 - 570 598; two tokens,
// in steps of four blocks, 387 | 466).
// Rows of any length that 32-bit offsets within a workgroup's 128 allow, by far (28672 columns left to the mat-vec: two 70B layers of Q8_0 at 5, 40 and 512 tokens 1264, 3008, 23941 us; here
// 762, 900, 3449).
bool mmq_q80_applicable(int type, int K, int T) { return type == T_Q8_0 && T >= 3 && K >= 256 && (K % 256) == 0 && K <= 65536; }

template <int SZ, int W, int S, int U> static void tiles_launch(Q80Args &a, hipStream_t st) {
    constexpr int R = 2 * SZ * W;
    int tiles = 0;
    for (int i = 0; i < a.n_seg; i++) { a.tile0[i] = tiles; tiles += (a.n_rows[i] + R - 1) / R; }
    hipLaunchKernelGGL((mmq_q80_tiles_kernel<SZ, W, S, U>), dim3((unsigned)tiles, (unsigned)((a.T + R - 1) / R)), dim3(256), 0, st, a);
}

// Up to two 32 x 32 workgroups a CU it is one wave's way through its row that counts, half as long in tiles of 16 (us, 16 | 32: 5632 x 2048, 40 tokens = 352 workgroups 9.6 | 12.9;
// 4096 x 14336, 100 = 512 48 | 74; 2048 x 2048, 320 = 640 13.1 | 13.0; 5632 x 2048, 100 = 704 14.1 | 13.3).  Four tiles of 32 a wave read half as much of LDS, but need 1.7 workgroups of 128 x 128 a CU and no more
// than a tenth more padding (us, one tile | four: 5632 x 2048, 1200 tokens = 440 workgroups 66 | 64; 4096 x 14336, 2000 = 512 470 | 415, 1200 = 320 283 | 330;
// 32000 x 2048, 320 = 750, a fifth more padding 92 | 100).
int mmq_q80_form(const int *n_rows, int n, int T) {
    const auto count = [&](int r) {
        long c = 0;
        for (int i = 0; i < n; i++) c += (n_rows[i] + r - 1) / r;
        return c * ((T + r - 1) / r);
    };
    const long c32 = count(32), c64 = count(64), c128 = count(128);
    return c32 <= 2L * num_cu() ? 16 : c128 * 10 >= 17L * num_cu() && c128 * 40 <= c64 * 11 ? 64 : 32;
}

hipError_t launch_mmq_q80_multi(const Q80Seg *sg, int n, int K, int T, const ActQuant &q, const float *resid, hipStream_t st) {
    if (!mmq_q80_applicable(T_Q8_0, K, T) || !q.qs0 || !q.d0 || n < 1 || n > 3) return hipErrorInvalidValue;
    for (int i = 0; i < n; i++)                                        // (16-byte requests of the codes and, in tiles of 16, of the scales)
        if (sg[i].row_bytes != sg[0].row_bytes || (((uintptr_t)sg[i].W | sg[i].row_bytes | (uintptr_t)q.qs0 | (uintptr_t)q.d0) & 15)) return hipErrorInvalidValue;
    Q80Args a{};
    a.row_bytes = sg[0].row_bytes; a.n_seg = n; a.K = K; a.T = T; a.aq = q.qs0; a.ad = q.d0; a.resid = resid;
    for (int i = 0; i < n; i++) { a.W[i] = sg[i].W; a.out[i] = sg[i].out; a.n_rows[i] = sg[i].n_rows; a.ld_out[i] = sg[i].ld_out; }
    switch (mmq_q80_form(a.n_rows, n, T)) {
        case 16: tiles_launch<16, 1, 3, 8>(a, st); break;
        case 64: tiles_launch<32, 2, 2, 4>(a, st); break;
        default: tiles_launch<32, 1, 3, 4>(a, st);
    }
    return hipGetLastError();
}

hipError_t launch_mmq_q80(const uint8_t *W, size_t row_bytes, int n_rows, int K, int T, const ActQuant &q, float *out, int ld_out,
                          const float *resid, hipStream_t st) {
    const Q80Seg sg{W, row_bytes, n_rows, out, ld_out};
    return launch_mmq_q80_multi(&sg, 1, K, T, q, resid, st);
}

}  // namespace mi355
