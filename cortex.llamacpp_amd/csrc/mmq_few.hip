// mmq_few.hip — the K-split contraction of 2 .. 64 tokens  Y[t][r] = dot(W[r,:], act_q8K[t,:])  (continuous-batching ticks, the short turn of a conversation):
// K-quant weights in their GGUF form, Q8_K activations, int8 matrix cores, the integer of ggml_vec_dot_q{4,5,6}_K_q8_K per (row, token, super-block).
//
// What bounds it: the weights, read once from HBM (0.56 .. 0.82 B each), and beside them the vector instructions per unit, ~200 for Q4_K and 280 for Q6_K at 48 tokens and their waits (two
// waves per SIMD; sixteen waves a CU are no faster); long rows of 37 tokens, 4096 x 14336, the activations' operands, which every workgroup reads: 290 MB from the L2 in 21 us.
// An 8B Q4_K_M model, kernel times (in front of them the 32 x 32 form of mmq.hip, whose waves had no load in flight while they computed and which left half of the CUs without a row
// tile): gate | up (66 MB) at 4 tokens 27.2 / 15.3 us, at 37 51.4 / 28.3; ffn_down at 4, Q4_K and Q6_K, 13.6 and 19.0, at 37 20.9 and 24.2; Q | K | V at 37 14.1 / 10.3; the head (431 MB) at 4
// 129 / 97, its rows on the host.
//   * A unit of work is 16 weight rows x one super-block (v_mfma_i32_16x16x32_i8: M = 16 tokens, N = 16 rows, K = the 32 weights of one scale group of Q4_K / Q5_K):
//     a 4096-row tensor is 256 row tiles, one per CU, and 16 tokens pad to 16, 37 to 48.
//   * One workgroup per CU walks its row tiles; its eight waves take a tile's super-blocks round-robin, and the weights of the next PD units - of the next tile
//     too - are in flight in registers while one is worked on.
//   * A wave asks for a unit as whole pieces of its rows, 144 (176, 208) consecutive bytes per row and super-block, and turns it into operands through LDS of its
//     own (a row's stride of 36, 44 or 52 words: no bank conflicts, no barrier).  Asked for as operands directly - 32 bytes of sixteen rows per request - every
//     128-byte line is asked for by four or five requests: gate | up of an 8B layer took 29 us that way.
//   * The activations come as operand blocks laid out by the quantiser (ActQuant::qf).  Read from rows of K bytes instead, sixteen lanes hit sixteen lines a power
//     of two apart: 34 us at 4 tokens, 43 at 16.  A wave meets the same super-blocks in every tile: up to 4096 columns and 48 tokens they stay in registers.
//   * From 17 tokens on (Q6_K from 9, Q5_K from 33) the groups' scales are folded into the weights, two codes a multiplication (Planes, few_planes): a super-block is two chains of MFMAs
//     of 64 weights, its integer one shift.  Before, an MFMA a group and four multiplications by its scale a tile: gate | up at 37 tokens 33.9 us, ffn_down of Q6_K 31.2, a prompt turn
//     of 37 tokens through eight layers of an 8B model 995 -> 903.
//   * To 8 and 4 tokens the operand's sixteen rows are two and four scale groups of a token (Act): half and a quarter of the multiplications by scales, the same integers.  Whole ticks of
//     eight layers of an 8B model, four conversations 790 -> 715 us (with PAIR 1 below), seven 797 -> 745.
//   * The eight partial sums of an output are added in wave order through LDS, so results do not depend on timing - and they are the sums the K-split
//     kernel of mmq.hip makes, bit for bit: an integer per super-block, the same fold, the same order.
#include <algorithm>

#include "kernels.h"

namespace mi355 {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int NW = 8, NT = 64 * NW;

__device__ __forceinline__ u32x4 ldg16(const void *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ u32x2 ldg8(const void *p) { return *reinterpret_cast<const u32x2 *>(p); }
__device__ __forceinline__ long as_long(u32x2 v) { return __builtin_bit_cast(long, v); }
__device__ __forceinline__ i32x4 mfma32(u32x2 a, u32x2 b, i32x4 c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(as_long(a), as_long(b), c, 0, 0, 0); }
__device__ __forceinline__ i32x4 mfma64(u32x4 a, u32x4 b, i32x4 c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0); }

// A unit, 16 rows x one super-block, as it is asked for: piece p = lane + 64 i is 16 bytes of row p / PIECES.  What of a piece's address is the lane's own stays in registers, the
// tile's and the super-block's share is scalar.  Tiles past the end of a tensor begin early enough to be whole (few_body), so rows are clamped only where there are fewer than sixteen
template <int TYPE, bool PAIR> struct Raw {
    static constexpr int PIECES = TYPE == T_Q4_K ? 9 : TYPE == T_Q5_K ? 11 : 13, N = (16 * PIECES + 63) / 64, LDS = N * 1024, STRIDE = 16 * PIECES;
    struct Where {                                           // PAIR: eight rows of two tensors, so whole addresses; else offsets from a scalar base
        unsigned o[N], u[N], d;                              // u: of a super-block (Q6_K: row planes ql, qh, scales, d, each with a step of its own)
        const uint8_t *b[PAIR ? N : 1], *bd;
    };
    static __device__ __forceinline__ void where(Where &w, const uint8_t *W, const uint8_t *W2, int rows, unsigned row_bytes, int nb, int lane) {
        const auto row = [&](int r) { return (unsigned)(PAIR ? (r & 7) < rows ? r & 7 : rows - 1 : r < rows ? r : rows - 1) * row_bytes; };
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int q = lane + 64 * i, p = q < STRIDE ? q : 0, r = p / PIECES, c = p - r * PIECES;    // (lanes past the unit: its first piece)
            w.o[i] = row(r) + (TYPE != T_Q6_K || c < 8 ? 16u * c : c < 12 ? (unsigned)nb * 128u + 16u * (c - 8) : (unsigned)nb * 192u);
            w.u[i] = TYPE != T_Q6_K ? (unsigned)STRIDE : c < 8 ? 128u : c < 12 ? 64u : 16u;
            if constexpr (PAIR) w.b[i] = (r < 8 ? W : W2) + w.o[i];
        }
        if constexpr (TYPE == T_Q6_K) {
            const int r = lane & 15;
            w.d = row(r) + (unsigned)nb * 208u;
            if constexpr (PAIR) w.bd = (r < 8 ? W : W2) + w.d;
        }
    }
    u32x4 v[N];
    uint32_t d16 = 0;                                        // Q6_K: the row's scale, which lies apart
    // at: what the tile's first row is away from the tensor's (bytes)
    __device__ __forceinline__ void load(const Where &w, const uint8_t *W, size_t at, int sb, int lane) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            if constexpr (TYPE == T_Q6_K) {
                const unsigned x = (unsigned)sb * w.u[i];
                v[i] = PAIR ? ldg16(w.b[PAIR ? i : 0] + at + x) : ldg16(W + at + (w.o[i] + x));
            } else {
                const size_t x = at + (unsigned)sb * (unsigned)STRIDE;
                v[i] = PAIR ? ldg16(w.b[PAIR ? i : 0] + x) : ldg16(W + x + w.o[i]);
            }
        }
        if constexpr (TYPE == T_Q6_K) {
            const size_t x = at + (unsigned)sb * 2u;
            d16 = *reinterpret_cast<const uint16_t *>(PAIR ? w.bd + x : W + x + w.d);
        }
    }
    __device__ __forceinline__ void put(uint8_t *lds, int lane) const {
#pragma unroll
        for (int i = 0; i < N; i++) *reinterpret_cast<u32x4 *>(lds + (lane + 64 * i) * 16) = v[i];
    }
};

// One lane's share of a unit as operands: row n = lane & 15, k-quarter kq = lane >> 4 of every MFMA step.
template <int TYPE> struct Frag;

// Q4_K / Q5_K: step J is scale group J (32 weights), the lane's 8 of them are bytes 8 kq .. of the group's 32-byte chunk (low / high nibbles)
template <> struct Frag<T_Q4_K> {
    static constexpr bool MINS = true;
    u32x4 h;
    u32x2 q[4];
    __device__ __forceinline__ void get(const uint8_t *lds, uint32_t, int n, int kq) {
        const uint8_t *b = lds + n * 144;
        h = ldg16(b);
#pragma unroll
        for (int c = 0; c < 4; c++) q[c] = ldg8(b + 16 + 32 * c + 8 * kq);
    }
    template <int J> __device__ __forceinline__ u32x2 codes() const {
        constexpr int sh = (J & 1) * 4;
        return u32x2{(q[J >> 1].x >> sh) & 0x0f0f0f0fu, (q[J >> 1].y >> sh) & 0x0f0f0f0fu};
    }
};
template <> struct Frag<T_Q5_K> {
    static constexpr bool MINS = true;
    u32x4 h;
    u32x2 q[4], qh;
    __device__ __forceinline__ void get(const uint8_t *lds, uint32_t, int n, int kq) {
        const uint8_t *b = lds + n * 176;
        h = ldg16(b);
        qh = ldg8(b + 16 + 8 * kq);
#pragma unroll
        for (int c = 0; c < 4; c++) q[c] = ldg8(b + 48 + 32 * c + 8 * kq);
    }
    template <int J> __device__ __forceinline__ u32x2 codes() const {
        constexpr int sh = (J & 1) * 4;
        return u32x2{((q[J >> 1].x >> sh) & 0x0f0f0f0fu) | (((qh.x >> J) & 0x01010101u) << 4),
                     ((q[J >> 1].y >> sh) & 0x0f0f0f0fu) | (((qh.y >> J) & 0x01010101u) << 4)};
    }
};
// Q6_K: step J is quarter J & 3 of half J >> 2 (low nibbles of ql for quarters 0 and 1, high for 2 and 3; two bits of qh), 16-groups 2 J and 2 J + 1
template <> struct Frag<T_Q6_K> {
    static constexpr bool MINS = false;
    u32x2 l[4], h[2];
    u32x4 sc;
    uint32_t d16;
    __device__ __forceinline__ void get(const uint8_t *lds, uint32_t d, int n, int kq) {
        const uint8_t *b = lds + n * 208;
#pragma unroll
        for (int i = 0; i < 4; i++) l[i] = ldg8(b + 32 * i + 8 * kq);
#pragma unroll
        for (int i = 0; i < 2; i++) h[i] = ldg8(b + 128 + 32 * i + 8 * kq);
        sc = ldg16(b + 192);
        d16 = d;
    }
    // the unsigned codes of 32 weights as they are
    template <int J> __device__ __forceinline__ u32x2 codes() const {
        constexpr int S = J >> 1, p = J & 1, n = S >> 1, nsh = (S & 1) * 4, up = 4 - nsh - 2 * p;
        u32x2 r;
#pragma unroll
        for (int i = 0; i < 2; i++) r[i] = ((l[2 * n + p][i] >> nsh) & 0x0f0f0f0fu) | ((up >= 0 ? h[n][i] << (up > 0 ? up : 0) : h[n][i] >> (up < 0 ? -up : 0)) & 0x30303030u);
        return r;
    }
};

// Group scales folded into the weights: of a unit's 64 weights of step S, a lane's sixteen as two int8 planes with  scale * code = (hi << SHIFT) + lo  (+ 128 in both planes of Q5_K),
// so that a super-block is two chains of MFMAs and one shift, and nothing is multiplied per output and group.  Two codes are multiplied at once, as bytes of a 16-bit lane:
//   Q4_K / Q5_K: scale = 8 s1 + s0, and a code times three bits stays in its byte (15 * 7, 31 * 7 = 217: the latter with 128 taken off, which the caller adds again as
//   128 * (8 + 1) times the sum of the activations);
//   Q6_K: (code - 32) * scale + 128 in 16 bits; its high byte is the one plane, its low one, the 128 taken off again, the other.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_u16(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t as_u32(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
template <int TYPE> struct Planes {
    static constexpr int SHIFT = TYPE == T_Q6_K ? 8 : 3;
    uint32_t s0[2], s1[2];                                   // Q4_K / Q5_K: the scales' low and high three bits, a byte a group
    __device__ __forceinline__ void scales(uint32_t sc_lo, uint32_t sc_hi) {
        s0[0] = sc_lo & 0x07070707u; s0[1] = sc_hi & 0x07070707u;
        s1[0] = (sc_lo >> 3) & 0x07070707u; s1[1] = (sc_hi >> 3) & 0x07070707u;
    }
    template <int S> __device__ __forceinline__ void step(const Frag<TYPE> &R, int kq, u32x4 &hi, u32x4 &lo) const {
        const u32x2 c[2] = {R.template codes<2 * S>(), R.template codes<2 * S + 1>()};
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const int J = 2 * S + g;
            if constexpr (TYPE == T_Q6_K) {                  // groups of sixteen: a lane's eight weights of 32 are of group 2 J + (kq >> 1)
                const int sc = __builtin_amdgcn_sbfe((int)R.sc[J >> 1], 8 * (2 * (J & 1) + (kq >> 1)), 8), off = 128 - 32 * sc;
                const u16x2 m = {(unsigned short)sc, (unsigned short)sc}, o = {(unsigned short)off, (unsigned short)off};
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t pe = as_u32(as_u16(c[g][i] & 0x00ff00ffu) * m + o), po = as_u32((as_u16(c[g][i]) >> (unsigned short)8) * m + o);
                    hi[2 * g + i] = __builtin_amdgcn_perm(po, pe, 0x07030501u);
                    lo[2 * g + i] = __builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u;
                }
            } else {
                const u16x2 w = as_u16(__builtin_amdgcn_perm(s1[J >> 2], s0[J >> 2], 0x0c040c00u + 0x00010001u * (J & 3)));
                const u16x2 m0 = {w.x, w.x}, m1 = {w.y, w.y};
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    hi[2 * g + i] = as_u32(as_u16(c[g][i]) * m1); lo[2 * g + i] = as_u32(as_u16(c[g][i]) * m0);
                    if constexpr (TYPE == T_Q5_K) { hi[2 * g + i] ^= 0x80808080u; lo[2 * g + i] ^= 0x80808080u; }
                }
            }
        }
    }
};

struct FewArgs {
    MMQSeg seg[3];
    int n_seg, K, T;
    const uint8_t *qf;
    // the output head (launch_mmq_few_head): rows for the host, [T][ld_out]; the workgroups' best logits of each row, and whose ticket is the last
    float *host, *best;
    int *best_row;
    unsigned *ticket;
    int32_t *win;
};

// One lane's activation operands of one super-block, as the quantiser laid them out (kernels.h FEW_BLOCK): token 16 * tile + (lane & 15) as the A operand - element
// pair (2 S, 2 S + 1) of scale groups per 16 bytes -, its block sums' two int8 planes, and the block scales of the four tokens whose results the lane holds.
// G = 2, 4 (to 8 and 4 tokens, one tile): the operand's row G t + g is token t with the weights of all scale groups but every G-th zeroed, so one MFMA makes the sums of G groups at
// once, and all of them are a lane's own 4 / G tokens': a G-th of the multiplications by scales.
template <int MT, int TYPE, int G> struct Act {
    u32x4 a[MT][4];
    u32x2 bh[MT], bl[MT];
    float yd[MT][4 / G];
    // (of the last tile's tokens past the batch, whose results are dropped, the last one's codes: other lines of the caches are not asked for)
    __device__ __forceinline__ void load_codes(const uint8_t *qf, int tile0, int nb, int sb, int lane, int s, int live) {
        const int m = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int tk = t == MT - 1 ? m / G < live ? m / G : live - 1 : m;
            a[t][s] = ldg16(qf + (size_t)((unsigned)((tile0 + t) * nb + sb) * (unsigned)FEW_BLOCK) + s * 1024 + (kq * 16 + tk) * 16);     // (the block is wave-uniform)
        }
    }
    __device__ __forceinline__ void load_rest(const uint8_t *qf, int tile0, int nb, int sb, int lane) {
        const int m = lane & 15, tk = m / G, kq = lane >> 4;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const uint8_t *p = qf + (size_t)((unsigned)((tile0 + t) * nb + sb) * (unsigned)FEW_BLOCK);
            const int o = tk * 16 + (kq & 1) * 8;
            bh[t] = ldg8(p + FEW_BH + o); bl[t] = ldg8(p + FEW_BL + o);
            if constexpr (G == 1) { const f32x4 y = *reinterpret_cast<const f32x4 *>(p + FEW_D + kq * 16); yd[t][0] = y.x; yd[t][1] = y.y; yd[t][2] = y.z; yd[t][3] = y.w; }
            else if constexpr (G == 2) { const f32x2 y = *reinterpret_cast<const f32x2 *>(p + FEW_D + kq * 8); yd[t][0] = y.x; yd[t][1] = y.y; }
            else yd[t][0] = *reinterpret_cast<const float *>(p + FEW_D + kq * 4);
        }
    }
    __device__ __forceinline__ void load(const uint8_t *qf, int tile0, int nb, int sb, int lane, int live) {
#pragma unroll
        for (int s = 0; s < 4; s++) load_codes(qf, tile0, nb, sb, lane, s, live);
        load_rest(qf, tile0, nb, sb, lane);
    }
    // G > 1, behind the loads: the other groups' weights zeroed
    __device__ __forceinline__ void mask(int lane) {
        if constexpr (G > 1) {
            const int g = lane & (G - 1), kq = lane >> 4;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                uint32_t lo, hi;                             // the 16 bytes' first and second 32 weights
                if constexpr (TYPE == T_Q6_K) {              // groups of sixteen: k-quarters 0, 1 and 2, 3 of each 32
                    const bool h = (kq >> 1) == (g & 1);
                    lo = h && (G == 2 || g < 2) ? ~0u : 0u; hi = h && (G == 2 || g >= 2) ? ~0u : 0u;
                } else {
                    const int x = G == 2 ? g : g - 2 * (s & 1);
                    lo = x == 0 ? ~0u : 0u; hi = x == 1 ? ~0u : 0u;
                }
                a[0][s] &= u32x4{lo, lo, hi, hi};
            }
        }
    }
};

// Scales in the weights, or on the sums of each group: 16 tokens of Q4_K and Q5_K need no fewer instructions with the former (us a pass of eight layers at 12 tokens, an 8B Q4_K_M and a 7B
// Q5_K_M model: 722 and 763 with it, 716 and 730 without; at 24, 37 and 48 of the former 806, 911 and 925, before 825, 994 and 1011)
template <int TYPE, int MT, int G> constexpr bool few_planes = G == 1 && (TYPE == T_Q6_K || MT > (TYPE == T_Q5_K ? 2 : 1));
// next(s): the operands of step s (4: the rest) are used, others may be asked for
template <int TYPE, int MT, int G, typename NEXT>
__device__ __forceinline__ void superblock(const Frag<TYPE> &R, const Act<MT, TYPE, G> &A, int kq, bool take, float (*facc)[4 / G], NEXT next) {
    constexpr int TPL = 4 / G;                               // a lane's tokens
    constexpr bool MINS = Frag<TYPE>::MINS;
    const i32x4 z = {0, 0, 0, 0};
    int isum[MT][TPL];
    // header of Q4_K / Q5_K: d, dmin, twelve bytes of 6-bit scales and mins
    uint32_t sc_lo = 0, sc_hi = 0, mn_lo = 0, mn_hi = 0;
    if constexpr (MINS) {
        sc_lo = R.h.y & 0x3f3f3f3fu; mn_lo = R.h.z & 0x3f3f3f3fu;
        sc_hi = (R.h.w & 0x0f0f0f0fu) | ((R.h.y >> 2) & 0x30303030u); mn_hi = ((R.h.w >> 4) & 0x0f0f0f0fu) | ((R.h.z >> 2) & 0x30303030u);
    }
    if constexpr (few_planes<TYPE, MT, G>) {
        Planes<TYPE> P;
        if constexpr (MINS) P.scales(sc_lo, sc_hi);
        i32x4 H[MT], L[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            H[t] = z; L[t] = z;
            if constexpr (TYPE == T_Q5_K) {                  // the sum of the token's activations: its sixteen block sums, in k-quarters 0 and 1
                const u32x2 one = kq < 2 ? u32x2{0x01010101u, 0x01010101u} : u32x2{0, 0};
                i32x4 v = mfma32(A.bh[t], one, z);
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] <<= 6;
                v = mfma32(A.bl[t], one, v);
#pragma unroll
                for (int r = 0; r < 4; r++) L[t][r] = __mul24(v[r], 128 * 9);
            }
        }
#define STEP(S)                                                                                                                      \
        {                                                                                                                            \
            u32x4 hi, lo;                                                                                                            \
            P.template step<S>(R, kq, hi, lo);                                                                                       \
            _Pragma("unroll") for (int t = 0; t < MT; t++) { H[t] = mfma64(A.a[t][S], hi, H[t]); L[t] = mfma64(A.a[t][S], lo, L[t]); } \
            next(S);                                                                                                                 \
        }
        STEP(0) STEP(1) STEP(2) STEP(3)
#undef STEP
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) isum[t][r] = (H[t][r] << Planes<TYPE>::SHIFT) + L[t][r];
    } else {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < TPL; r++) isum[t][r] = 0;
#define HALF(J, t) ((J & 1) ? u32x2{A.a[t][J >> 1].z, A.a[t][J >> 1].w} : u32x2{A.a[t][J >> 1].x, A.a[t][J >> 1].y})
#define BOTH(S) ({ const u32x2 b0_ = R.template codes<2 * (S)>(), b1_ = R.template codes<2 * (S) + 1>(); u32x4{b0_.x, b0_.y, b1_.x, b1_.y}; })
        if constexpr (MINS) {
            const auto scale = [&](int J) { return (int)(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff); };
            if constexpr (G == 1) {
#define STEP(J)                                                                                              \
            {                                                                                                \
                const int sc = scale(J);                                                                     \
                const u32x2 b = R.template codes<J>();                                                       \
                _Pragma("unroll") for (int t = 0; t < MT; t++) {                                             \
                    const i32x4 I = mfma32(HALF(J, t), b, z);                                                \
                    _Pragma("unroll") for (int r = 0; r < 4; r++) isum[t][r] = __mul24(I[r], sc) + isum[t][r]; \
                    if constexpr (MT > 1) { _Pragma("unroll") for (int r = 0; r < 4; r++) asm volatile("" : "+v"(isum[t][r])); }   /* (the sums are reassociated otherwise, every product alive) */ \
                }                                                                                            \
            }
            STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5) STEP(6) STEP(7)
#undef STEP
            } else if constexpr (G == 2) {
#define STEP(S)                                                                                              \
            {                                                                                                \
                const i32x4 I = mfma64(A.a[0][S], BOTH(S), z);                                               \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[0][r >> 1] = __mul24(I[r], scale(2 * S + (r & 1))) + isum[0][r >> 1]; \
            }
            STEP(0) STEP(1) STEP(2) STEP(3)
#undef STEP
            } else {
#define STEP(C)                                                                                              \
            {                                                                                                \
                const i32x4 I = mfma64(A.a[0][2 * C + 1], BOTH(2 * C + 1), mfma64(A.a[0][2 * C], BOTH(2 * C), z)); \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[0][0] = __mul24(I[r], scale(4 * C + r)) + isum[0][0]; \
            }
            STEP(0) STEP(1)
#undef STEP
            }
        } else {
            // the raw codes, 16-group by 16-group, the signed scale on the four results
            const auto scale = [&](int j) { return (int)(int8_t)((R.sc[j >> 2] >> (8 * (j & 3))) & 0xff); };
            if constexpr (G == 2) {
#define STEP(J)                                                                                              \
            {                                                                                                \
                const i32x4 I = mfma32(HALF(J, 0), R.template codes<J>(), z);                                   \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[0][r >> 1] = __mul24(I[r], scale(2 * J + (r & 1))) + isum[0][r >> 1]; \
            }
            STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5) STEP(6) STEP(7)
#undef STEP
            } else {
#define STEP(S)                                                                                              \
            {                                                                                                \
                const i32x4 I = mfma64(A.a[0][S], BOTH(S), z);                                               \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[0][0] = __mul24(I[r], scale(4 * S + r)) + isum[0][0]; \
            }
            STEP(0) STEP(1) STEP(2) STEP(3)
#undef STEP
            }
        }
#undef HALF
#undef BOTH
#pragma unroll
        for (int s = 0; s < 4; s++) next(s);
    }
    // the block sums: against the mins (min j meets sums 2 j and 2 j + 1), or for the code's "- 32" against the scales; k-quarters 0 and 1 hold them, 2 and 3 are zero
    if constexpr (MINS) {
        const uint32_t mw = kq == 0 ? mn_lo : mn_hi;
        u32x2 bm = {__builtin_amdgcn_perm(0, mw, 0x01010000u), __builtin_amdgcn_perm(0, mw, 0x03030202u)};
        if (kq >= 2) bm = u32x2{0, 0};
        const uint32_t dw = take ? R.h.x : 0u;
        const float dd = h2f((uint16_t)(dw & 0xffff)), dm = h2f((uint16_t)(dw >> 16));
#pragma unroll
        for (int t = 0; t < MT; t++) {
            i32x4 ms = mfma32(A.bh[t], bm, z);
#pragma unroll
            for (int r = 0; r < 4; r++) ms[r] <<= 6;
            ms = mfma32(A.bl[t], bm, ms);
#pragma unroll
            for (int r = 0; r < TPL; r++) facc[t][r] += (dd * A.yd[t][r]) * (float)isum[t][r] - (dm * A.yd[t][r]) * (float)ms[G * r];
        }
    } else {
        const float dd = h2f((uint16_t)(take ? R.d16 : 0u));
        if constexpr (G > 1) {
            u32x2 bm = kq == 0 ? u32x2{R.sc.x, R.sc.y} : u32x2{R.sc.z, R.sc.w};
            if (kq >= 2) bm = u32x2{0, 0};
            i32x4 ms = mfma32(A.bh[0], bm, z);
#pragma unroll
            for (int r = 0; r < 4; r++) ms[r] <<= 6;
            ms = mfma32(A.bl[0], bm, ms);
#pragma unroll
            for (int r = 0; r < TPL; r++) isum[0][r] -= 32 * ms[G * r];
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < TPL; r++) facc[t][r] += (dd * A.yd[t][r]) * (float)isum[t][r];
    }
    next(4);
}

// LDS of a workgroup: every wave's staging area (NP units), then the sets of partial sums [wave][unit][tile * 4 / G + r][lane]
template <int TYPE, int NP> constexpr int few_stage = NW * NP * Raw<TYPE == 0 ? T_Q6_K : TYPE, false>::LDS;
template <int MT, int NP> constexpr int few_sets = MT * NP == 1 ? 2 : 1;  // two in turn: one barrier per tile
template <int TYPE, int MT, int G, int NP> constexpr int few_lds = few_stage<TYPE, NP> + few_sets<MT, NP> * NW * NP * MT * (1024 / G);

// CN > 0: every wave has (up to) CN <= PD super-blocks of a tile and keeps their activation operands in registers across tiles.  CN = 0: any number, the operands
// are read (from the caches) a unit ahead.
// out = silu(gate . x) * (up . x): PAIR 1, a tile is eight rows of ffn_gate and the same eight of ffn_up, one unit; PAIR 2, sixteen rows of each, two units against the same
// activation operands.  14336 rows are seven tiles a CU of the first kind and three and a half, four for half of them, of the second; but where the operands are read again for every tile
// the first reads them twice as often (few_pair).
// HEAD: see mmq_few_head_kernel
constexpr int HEAD_RUN = 4;                                  // row tiles whose results are stored to the host together, a wave's width of rows (two: 16 rows 20 us slower; eight: 4 and 16 rows 8 us)
template <int MT> constexpr int head_lds = 2 * 16 * MT * HEAD_RUN * 64;
template <int TYPE, int MT, int G, int PAIR, int PD, int CN, bool HEAD = false>
__device__ __forceinline__ void few_body(const FewArgs &a, const MMQSeg &sg, int tile, int n_blocks, uint8_t *smem, int stage_bytes) {
    constexpr int TR = PAIR == 1 ? 8 : 16, TPL = 4 / G, NP = PAIR == 2 ? 2 : 1;           // a tile's rows (of each tensor), a lane's tokens of a token tile, a tile's units
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, kq = lane >> 4;
    const int nb = a.K >> 8, T = a.T;
    int tiles = (sg.n_rows + TR - 1) / TR;
    if constexpr (HEAD) {                                    // (a run of neighbours)
        const int b = tile, all = tiles, each = n_blocks;
        tile = (int)((long long)all * b / each); tiles = (int)((long long)all * (b + 1) / each);
        n_blocks = 1;
    }
    const int tile0 = tile;
    const int row_max = sg.n_rows > TR ? sg.n_rows - TR : 0; // a tile's first row at most: the last tile begins early enough to be whole, and stores the rows that are its own
    uint8_t *stage = smem + wave * (NP * Raw<TYPE, PAIR == 1>::LDS);
    float *part = reinterpret_cast<float *>(smem + stage_bytes);
    // operands that are read again stay a unit or two ahead
    constexpr int PA = CN > 0 ? CN : MT == 1 ? 2 : 1;
    static_assert(CN == 0 || MT <= 3, "operands of four token tiles are not kept");
    static_assert(G == 1 || MT == 1, "one token tile");
    const int cn = CN > 0 ? CN : (nb + NW - 1) / NW;
    float facc[NP][MT][TPL];
    auto clear = [&]() {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < TPL; r++) facc[p][t][r] = 0.0f;
    };
    clear();
    typedef Raw<TYPE, PAIR == 1> RawT;
    typedef Act<MT, TYPE, G> ActT;
    typename RawT::Where where;
    RawT::where(where, sg.W, PAIR == 1 ? a.seg[1].W : nullptr, sg.n_rows < TR ? sg.n_rows : TR, (unsigned)sg.row_bytes, nb, lane);
    RawT R[PD][NP];
    ActT A[PA];
    // the unit the next request is for; past the end it stays on the last one
    int l_tile = tile, l_i = 0;
    auto request = [&](RawT (&r)[NP]) {
        const int row0 = l_tile * TR < row_max ? l_tile * TR : row_max;
        const int sb = wave + NW * l_i < nb ? wave + NW * l_i : nb - 1;
        r[0].load(where, sg.W, (size_t)row0 * sg.row_bytes, sb, lane);
        if constexpr (NP == 2) r[1].load(where, a.seg[1].W, (size_t)row0 * sg.row_bytes, sb, lane);
        if (l_i + 1 < cn) l_i++;
        else if (l_tile + n_blocks < tiles) { l_tile += n_blocks; l_i = 0; }
    };
    const int live = T - 16 * (MT * (int)blockIdx.y + MT - 1) < 1 ? 1 : T - 16 * (MT * (int)blockIdx.y + MT - 1);
    const auto act_sb = [&](int i) { const int sb = wave + NW * i; return sb < nb ? sb : nb - 1; };
    // an output of a finished tile: element e = tid + NT j of [tile * TPL + r][lane].  Its residual is requested a tile ahead, in front of the weights that follow
    constexpr int NS = MT * TPL * 64, NE = (NS + NT - 1) / NT;
    float rv[NE];
    auto token = [&](int e) { const int tr = e >> 6; return (tr / TPL) * 16 + TPL * ((e & 63) >> 4) + tr % TPL; };
    auto place = [&](int e, int row_tile, size_t &o) {
        const int gt = blockIdx.y * 16 * MT + token(e), row0 = row_tile * TR < row_max ? row_tile * TR : row_max, row = row0 + (e & (TR - 1));
        o = (size_t)gt * sg.ld_out + row;
        return e < NS && gt < T && row >= row_tile * TR && row < sg.n_rows && (e & 15) < TR;
    };
    auto residual = [&](int row_tile) {
        if constexpr (PAIR == 0) if (sg.resid) {
#pragma unroll
            for (int j = 0; j < NE; j++) { size_t o; const bool in = place(tid + NT * j, row_tile, o); rv[j] = sg.resid[in ? o : 0]; }
        }
    };
    int set = 0;
    // HEAD: results wait in LDS for the other tiles of their run, [run parity][token][row]; a thread's outputs are all of one token
    float *const run = part + few_sets<MT, NP> * NW * NP * NS;
    float top = -INFINITY;
    int top_row = 0x7fffffff;
    auto to_host = [&](int done) {                           // the run that ends in front of `done`, behind a barrier
        if (!a.host) return;
        const int k0 = (done - tile0 - 1) / HEAD_RUN * HEAD_RUN, n = (done - tile0 - k0) * 16;
        const float *const r0 = run + (k0 / HEAD_RUN & 1) * 16 * MT * (HEAD_RUN * 16);
        const int row0 = (tile0 + k0) * 16, rows = sg.n_rows - row0 < n ? sg.n_rows - row0 : n;
        for (int t = wave; t < T; t += NW)
            if (lane < rows) a.host[(size_t)t * sg.ld_out + row0 + lane] = r0[t * (HEAD_RUN * 16) + lane];
    };
    auto finish = [&](int row_tile) {
        float *ps = part + set * (NW * NP * NS);
        set ^= few_sets<MT, NP> - 1;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < TPL; r++) ps[(wave * NP + p) * NS + (t * TPL + r) * 64 + lane] = facc[p][t][r];
        __syncthreads();
        if constexpr (HEAD) if (row_tile > tile0 && (row_tile - tile0) % HEAD_RUN == 0) to_host(row_tile);
#pragma unroll
        for (int j = 0; j < NE; j++) {
            const int e = tid + NT * j;
            size_t o;
            if (place(e, row_tile, o)) {
                float sum = 0.0f, sum2 = 0.0f;
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    sum += ps[w * NP * NS + e];
                    if constexpr (PAIR) sum2 += ps[PAIR == 1 ? w * NS + e + 8 : (w * NP + 1) * NS + e];
                }
                if constexpr (PAIR) sg.out[o] = (sum / (1.0f + expf(-sum))) * sum2;
                else sg.out[o] = sg.resid ? rv[j] + sum : sum;
                if constexpr (HEAD) {
                    const int k = row_tile - tile0, gt = token(e), row = (int)(o - (size_t)gt * sg.ld_out);
                    run[((k / HEAD_RUN & 1) * 16 * MT + gt) * (HEAD_RUN * 16) + (k % HEAD_RUN) * 16 + (row - row_tile * 16)] = sum;
                    if (sum > top || (sum == top && row < top_row)) { top = sum; top_row = row; }
                }
            }
        }
        if constexpr (few_sets<MT, NP> == 1) __syncthreads();
        clear();
    };
    residual(tile);
#pragma unroll
    for (int i = 0; i < PA; i++) A[i].load(a.qf, blockIdx.y * MT, nb, act_sb(i < cn ? i : 0), lane, live);
    // (the requests in the order of their use, none moved past another: a wait for one slot must not be a wait for the others)
#pragma unroll
    for (int u = 0; u < PD; u++) { __builtin_amdgcn_sched_barrier(0); request(R[u]); __builtin_amdgcn_sched_barrier(0); }
    static_assert(CN == 0 || PD % CN == 0, "a slot belongs to one super-block of the tile");
    static_assert(CN > 0 || PD % PA == 0, "activation slots turn with the weight slots");
    if constexpr (CN > 0) {
#pragma unroll
        for (int i = 0; i < PA; i++) A[i].mask(lane);
    }
    int i = 0;
    auto unit = [&](RawT (&r)[NP], ActT &x, int i) {
        const bool take = wave + NW * i < nb;                              // (a tile of nb super-blocks does not divide by the waves: the last unit's share is multiplied by a zero scale, not branched around)
        uint32_t d16[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) { r[p].put(stage + p * RawT::LDS, lane); d16[p] = r[p].d16; }
        __builtin_amdgcn_sched_barrier(0);                                 // (a wave's LDS accesses are made in order)
        request(r);                                                        // the slot's next unit, in flight across this one's arithmetic
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (CN == 0) x.mask(lane);
        const int j = i + PA, then = act_sb(j < cn ? j : j - cn < cn ? j - cn : 0);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            Frag<TYPE> f;
            f.get(stage + p * RawT::LDS, d16[p], n, kq);
            superblock<TYPE, MT, G>(f, x, kq, take, facc[p], [&](int s) {
                if (CN > 0 || p < NP - 1) return;
                if (s < 4) x.load_codes(a.qf, blockIdx.y * MT, nb, then, lane, s, live); else x.load_rest(a.qf, blockIdx.y * MT, nb, then, lane);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_wave_barrier();
    };
    const int mine = (tiles - tile + n_blocks - 1) / n_blocks, S = mine * cn;
    for (int s = 0; s < S; s += PD) {
#pragma unroll
        for (int u = 0; u < PD; u++) {
            if (CN > 0 ? u % (CN > 0 ? CN : 1) == 0 && s + u >= S : s + u >= S) goto done;
            unit(R[u], A[CN > 0 ? u % (CN > 0 ? CN : 1) : u % PA], CN > 0 ? u % (CN > 0 ? CN : 1) : i);
            if (CN > 0 ? (u + 1) % (CN > 0 ? CN : 1) == 0 : ++i == cn) { i = 0; finish(tile); tile += n_blocks; residual(tile < tiles ? tile : 0); }
        }
    }
done:
    if constexpr (HEAD) {
        __syncthreads();
        if (tiles > tile0) to_host(tiles);
        // the best of the workgroup's rows: a token's results are sixteen neighbouring lanes'
        static_assert(NE == 1, "a thread's results are of one token");
        const auto better = [&](float v, int r) { if (v > top || (v == top && r < top_row)) { top = v; top_row = r; } };
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) { const float v = __shfl_xor(top, o, 64); const int r = __shfl_xor(top_row, o, 64); better(v, r); }
        const int gt = token(tid), blocks = (int)gridDim.x;
        if (tid < NS && (lane & 15) == 0 && gt < T) {
            __hip_atomic_store(a.best + gt * blocks + blockIdx.x, top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.best_row + gt * blocks + blockIdx.x, top_row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // (the write-through stores have left before the ticket is taken)
        int *const last = reinterpret_cast<int *>(smem);
        __syncthreads();
        if (tid == 0) {
            const unsigned t = __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *last = t == (unsigned)blocks - 1u;
            if (*last) __hip_atomic_store(a.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // re-armed for the next launch
        }
        __syncthreads();
        if (!*last) return;
        for (int t = wave; t < T; t += NW) {
            top = -INFINITY; top_row = 0x7fffffff;
            for (int b = lane; b < blocks; b += 64)
                better(__hip_atomic_load(a.best + t * blocks + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __hip_atomic_load(a.best_row + t * blocks + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) { const float v = __shfl_xor(top, o, 64); const int r = __shfl_xor(top_row, o, 64); better(v, r); }
            if (lane == 0) a.win[t] = top_row;
        }
    }
}

// TYPE: the segments' common type, or 0 where they differ (Q | K | V of a layer whose attn_v is wider)
template <int TYPE, int MT, int G, int PAIR, int PD, int CN>
__global__ __launch_bounds__(NT, 2) void mmq_few_kernel(const FewArgs a) {
    constexpr int NP = PAIR == 2 ? 2 : 1;
    __shared__ __attribute__((aligned(16))) uint8_t smem[few_lds<TYPE, MT, G, NP>];
    int s = 0;
    if constexpr (!PAIR) {
        if (a.n_seg > 1 && (int)blockIdx.x >= a.seg[1].tile0) s = 1;
        if (a.n_seg > 2 && (int)blockIdx.x >= a.seg[2].tile0) s = 2;
    }
    const int first = (int)blockIdx.x - a.seg[s].tile0, n_blocks = (s + 1 < a.n_seg && !PAIR ? a.seg[s + 1].tile0 : (int)gridDim.x) - a.seg[s].tile0;
    if constexpr (TYPE != 0) few_body<TYPE, MT, G, PAIR, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>);
    else switch (a.seg[s].type) {
        case T_Q4_K: few_body<T_Q4_K, MT, G, PAIR, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        case T_Q5_K: few_body<T_Q5_K, MT, G, PAIR, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        case T_Q6_K: few_body<T_Q6_K, MT, G, PAIR, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        default: break;
    }
}

// The output head of a tick: a workgroup takes a run of neighbouring row tiles, and stores the results of HEAD_RUN of them at a time - 256 consecutive bytes a token - to the
// host's rows while its weights stream: PCIe bounds it from a dozen rows on.  The rows' arg-max is made of what the threads hold anyway.  128256 rows of 4096 columns (Q6_K), us, here /
// the head, the arg-max and a launch that copies the rows one behind the other: 4 tokens 97 / 99 + 10 + 38, 16 tokens 205 / 104 + 19 + 149.
template <int TYPE, int MT, int G, int CN>
__global__ __launch_bounds__(NT, 2) void mmq_few_head_kernel(const FewArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[few_lds<TYPE, MT, G, 1> + head_lds<MT>];
    few_body<TYPE, MT, G, 0, 4, CN, true>(a, a.seg[0], (int)blockIdx.x, (int)gridDim.x, smem, few_stage<TYPE, 1>);
}
template <int TYPE>
void few_head(const FewArgs &a, int blocks, hipStream_t st) {
    const int cn = ((a.K >> 8) + NW - 1) / NW;
#define GO(MT, G, CN) hipLaunchKernelGGL((mmq_few_head_kernel<TYPE, MT, G, CN>), dim3((unsigned)blocks), dim3(NT), 0, st, a)
#define GO_CN(MT, G) do { if (cn == 1) GO(MT, G, 1); else if (cn == 2) GO(MT, G, 2); else GO(MT, G, 0); } while (0)
    if (a.T <= 4) GO_CN(1, 4); else if (a.T <= 8) GO_CN(1, 2); else if (a.T <= 16) GO_CN(1, 1); else GO_CN(2, 1);
#undef GO_CN
#undef GO
}

// The form of a gate | up launch: the operands of up to 48 tokens stay in registers to 4096 columns, and to eight tokens they are few.  us a pass, PAIR 1 / 2: three layers of 5120 columns
// at 4 and 12 tokens 395 / 437, 492 / 497, two of 8192 at 4, 12, 24 and 40 625 / 683, 747 / 736, 986 / 942, 790 / 752; 37.2 / 34.1 a launch of 14336 x 4096 at 37
int few_pair(int K, int T) { return T <= 8 || (K <= 2 * NW * 256 && T <= 48) ? 1 : 2; }

template <int TYPE, int PAIR>
void few_type(const FewArgs &a, int blocks, hipStream_t st) {
    const int cn = ((a.K >> 8) + NW - 1) / NW;
    // four units of weights in flight per wave: 74 KB per CU (three and four token tiles: two, their operands take the registers)
#define GO(MT, G, PD, CN) hipLaunchKernelGGL((mmq_few_kernel<TYPE, MT, G, PAIR, PD, CN>), dim3((unsigned)blocks, (unsigned)((a.T + 16 * MT - 1) / (16 * MT))), dim3(NT), 0, st, a)
#define GO_CN(MT, G) do { if (cn == 1) GO(MT, G, 4, 1); else if (cn == 2) GO(MT, G, 4, 2); else GO(MT, G, 4, 0); } while (0)
    if constexpr (PAIR == 2) {
        if (a.T <= 16) GO(1, 1, 2, 0); else if (a.T <= 32) GO(2, 1, 2, 0); else if (a.T <= 48) GO(3, 1, 1, 0); else GO(4, 1, 1, 0);
    } else if (a.T <= 4) GO_CN(1, 4);
    else if (a.T <= 8) GO_CN(1, 2);
    else if (a.T <= 16) { if (cn == 1) GO(1, 1, 4, 1); else if (cn == 2) GO(1, 1, 4, 2); else if constexpr (PAIR == 0) GO(1, 1, 4, 0); }
    else if (a.T <= 32) { if (cn == 1) GO(2, 1, 4, 1); else if (cn == 2) GO(2, 1, 4, 2); else if constexpr (PAIR == 0) GO(2, 1, 4, 0); }
    else if (a.T <= 48) { if (cn == 1) GO(3, 1, 2, 1); else if (cn == 2) GO(3, 1, 2, 2); else if constexpr (PAIR == 0) GO(3, 1, 2, 0); }
    else if constexpr (PAIR == 0) GO(4, 1, 2, 0);
#undef GO_CN
#undef GO
}

constexpr int FEW_PAIR_K = 1280;

}  // namespace

// Whether a launch of T tokens is the faster one here (the sums are the same either way; us, here against the K-split kernel of mmq.hip):
//   * to 16 tokens: 4.2 / 6.1 (2048 x 2048) .. 62 / 100 (128256 x 4096), Q6_K 104 / 139;
//   * to 48: as long as the row tiles fill their rounds of CUs - 320 of 512 do not: 5120 x 5120 14.3 / 10.8 at 17 tokens, 17.9 / 16.4 at 33 - and, for Q6_K, whose units
//     take twice the instructions, there is but one round: 4096 x 4096 10.8 / 13.3, but 6144 x 4096 15.6 / 14.1 and 152064 x 3584 270 / 242;
//   * to 64, where the operands of four token tiles leave two units in flight: gate | up, 42 / 50 (14336 x 4096), and long rows, 32.7 / 39.5 (4096 x 14336) - but 13.5 / 12.7
//     (4096 x 4096), 112 / 77 (8192 x 28672: 512 row tiles), 318 / 217 (152064 x 3584), and Q6_K never, 549 / 233.
// Two tokens, from rows of FEW_PAIR_K columns on.  The mat-vec's sums of two are the one-token step's only for Q6_K and while no two waves share a row, so a pair of conversations and either alone
// are as far apart there as any two orders of a sum are (8B and 7B: logits 0.010).  us a tick of two conversations and a turn of two tokens, here / the mat-vec: eight 8B Q4_K_M layers
// 677 / 885, 648 / 805, eight 7B Q5_K_M layers 654 / 870, 627 / 847, six layers of 2048 and 5632 columns, Q4_K_M 313 / 384, 297 / 386; of 1280 and 3584 columns a tick 293, of three 305.  Of
// shorter rows launches are latency (1024 and 2816 columns, two 328, three 303; 512 and 1536 313, 288), and they stay with the mat-vec, whose sums come closest to the single step's.
bool mmq_few_pair(int type, int K, int T, const ActQuant &q) { return T == 2 && q.qf && (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && (K & 255) == 0 && K >= FEW_PAIR_K; }
bool mmq_few_takes(const MMQSeg *segs, int n_seg, int K, int T, const ActQuant &q, bool swiglu) {
    if (!q.qf || T > FEW_MAX_T) return false;
    if (T <= 16) return true;
    int tiles = 0, q6 = 0;
    for (int i = 0; i < n_seg; i++) { if (!swiglu || i == 0) tiles += (segs[i].n_rows + 15) / 16; q6 += segs[i].type == T_Q6_K; }
    const bool one_round = tiles <= num_cu();
    if (T <= 48) return q6 == n_seg ? one_round : one_round || 2 * tiles >= 3 * num_cu();
    return q6 == 0 && (swiglu || (one_round && K > 4096));
}

// segs as launch_mmq_ksplit_multi's (which comes here where mmq_few_takes says so): up to three tensors sharing the activation, or {gate, up} of one type and shape with swiglu
hipError_t launch_mmq_few(const MMQSeg *segs, int n_seg, int K, int T, const ActQuant &q, bool swiglu, hipStream_t st) {
    if (!q.qf || T > FEW_MAX_T) return hipErrorInvalidValue;
    FewArgs a{};
    a.n_seg = n_seg; a.K = K; a.T = T;
    a.qf = q.qf;
    // one workgroup per CU where there are more row tiles than that.  Segments of different types: as few rounds as a Q6_K tile of one and a half others' allow (Q | K | V with a
    // Q6_K attn_v, 256 + 64 + 64 tiles, us at 4 and 16 tokens: 12.1, 12.2 where every tensor gets its share by rows - V's tiles two to a workgroup - here 8.6, 9.6); the CUs left over by rows
    const int ns = swiglu ? 1 : n_seg, pair = swiglu ? few_pair(K, T) : 0, tr = pair == 1 ? 8 : 16;
    int tiles = 0, type = segs[0].type, t[3] = {0, 0, 0}, n[3] = {0, 0, 0};
    for (int i = 0; i < ns; i++) { tiles += t[i] = (segs[i].n_rows + tr - 1) / tr; if (segs[i].type != type) type = 0; }
    const int cap = std::max(ns, std::min(tiles, num_cu()));
    const auto cost = [&](int i) { return segs[i].type == T_Q6_K ? 3 : 2; };
    for (int budget = 3;; budget++) {
        int sum = 0;
        for (int i = 0; i < ns; i++) { const int each = std::max(1, budget / cost(i)); sum += n[i] = (t[i] + each - 1) / each; }
        if (sum <= cap || budget > 3 * tiles) break;
    }
    for (int left = cap - n[0] - n[1] - n[2]; left > 0; left--) {
        int k = 0;
        for (int i = 1; i < ns; i++) if ((long long)t[i] * cost(i) * n[k] > (long long)t[k] * cost(k) * n[i]) k = i;
        if (n[k] >= t[k]) break;
        n[k]++;
    }
    int blocks = 0;
    for (int i = 0; i < n_seg; i++) {
        a.seg[i] = segs[i];
        a.seg[i].tile0 = blocks;
        if (i < ns) blocks += n[i];
    }
    if (swiglu) switch (type) {
        case T_Q4_K: if (pair == 1) few_type<T_Q4_K, 1>(a, blocks, st); else few_type<T_Q4_K, 2>(a, blocks, st); break;
        case T_Q5_K: if (pair == 1) few_type<T_Q5_K, 1>(a, blocks, st); else few_type<T_Q5_K, 2>(a, blocks, st); break;
        case T_Q6_K: if (pair == 1) few_type<T_Q6_K, 1>(a, blocks, st); else few_type<T_Q6_K, 2>(a, blocks, st); break;
        default: return hipErrorInvalidValue;
    } else switch (type) {
        case T_Q4_K: few_type<T_Q4_K, 0>(a, blocks, st); break;
        case T_Q5_K: few_type<T_Q5_K, 0>(a, blocks, st); break;
        case T_Q6_K: few_type<T_Q6_K, 0>(a, blocks, st); break;
        default: few_type<0, 0>(a, blocks, st); break;
    }
    return hipGetLastError();
}

static int head_blocks(int n_rows) { return std::min((n_rows + 15) / 16, num_cu()); }
size_t mmq_few_head_scratch() { return 1 + 2 * (size_t)HEAD_MAX_T * (size_t)num_cu(); }
// Over its whole range the faster one, also where 17 rows and more of Q6_K are the K-split kernel's otherwise (mmq_few_takes), and where the rows stay on the device: us a call of one
// layer and the head, here / that kernel or mmq_few_kernel with the arg-max, and the copy, behind it
//   128256 x 4096, rows on the host    3: 219 / 252, 8: 245 / 317, 16: 352 / 424, 17: 390 / 482, 24: 477 / 564, 32: 572 / 668      left on the device   3: 221 / 227, 16: 260 / 274, 17: 310 / 329, 32: 340 / 365
//   32000 x 4096                       3: 152 / 163, 8: 173 / 188, 16: 214 / 237, 17: 245 / 268, 24: 271 / 302, 32: 315 / 346                           3: 148 / 155, 16: 185 / 199, 17: 216 / 227, 32: 255 / 267
//   32000 x 2048                       3: 115 / 119, 8: 131 / 144, 16: 167 / 186, 17: 182 / 197, 24: 210 / 227, 32: 251 / 273                           3: 108 / 111, 16: 133 / 147, 17: 148 / 156, 32: 186 / 195
bool mmq_few_head_takes(int type, int K, int T, const ActQuant &q) {
    return q.qf && (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && (K & 255) == 0 && (T >= 3 || mmq_few_pair(type, K, T, q)) && T <= HEAD_MAX_T;
}
hipError_t launch_mmq_few_head(const MMQSeg &seg, int K, int T, const ActQuant &q, float *host, float *scratch, int32_t *win, hipStream_t st) {
    if (!mmq_few_head_takes(seg.type, K, T, q) || !scratch || !win || seg.resid || seg.n_rows < 1) return hipErrorInvalidValue;
    FewArgs a{};
    a.n_seg = 1; a.K = K; a.T = T;
    a.qf = q.qf;
    a.seg[0] = seg;
    a.seg[0].tile0 = 0;
    const int blocks = head_blocks(seg.n_rows);
    a.host = host; a.win = win;
    a.ticket = reinterpret_cast<unsigned *>(scratch);
    a.best = scratch + 1;
    a.best_row = reinterpret_cast<int *>(a.best + (size_t)HEAD_MAX_T * num_cu());
    switch (seg.type) {
        case T_Q4_K: few_head<T_Q4_K>(a, blocks, st); break;
        case T_Q5_K: few_head<T_Q5_K>(a, blocks, st); break;
        default: few_head<T_Q6_K>(a, blocks, st); break;
    }
    return hipGetLastError();
}

}  // namespace mi355
