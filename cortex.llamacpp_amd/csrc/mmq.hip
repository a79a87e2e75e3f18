// mmq.hip — batched prefill contraction  Y[t][r] = dot(W[r,:], act_q8K[t,:])  on the MFMA matrix cores.
//
// Stands in for ggml's mul_mat_q / the CPU backend's chunked mul_mat for prompt processing,
// reached from the reference through llama_decode with n_tokens > 1 (src/llama_server_context.cc:1568-1607, 1635).
//
// Integer-exact by construction, and MFMA-bound rather than VALU-bound:
//   ggml_vec_dot_q{4,5,6}_K_q8_K computes, per (row, token, super-block of 256),   isum = sum_g sc_g * sum_{k in g} q_k a_k
//   with 6-bit (Q4_K/Q5_K, groups of 32) or int8 (Q6_K, groups of 16) group scales sc_g.  Applying sc_g to the int32
//   MFMA result costs one multiply-add per OUTPUT per group (16 VALU ops per MFMA — as long as the MFMA itself).  Here
//   the scale is folded into the WEIGHT instead:  p_k = sc_g * q_k  (10..13 bits) is split into two int8 planes
//   p_k = 2^S * hi_k + lo_k, and  isum = 2^S * (hi . a) + (lo . a)  is two MFMA accumulation chains over the whole
//   super-block with nothing in between.  The split is exact, so isum is bit-identical to the CPU's integer.
//   The expansion costs VALU work per WEIGHT (not per output) and is amortised over the wave's token tiles.
//   * Q4_K / Q5_K: q in [0,15] / [0,31], sc in [0,63]: S = 5, hi <= 29 / 61, lo <= 31.  The "mins" term
//     msum = sum_j m_j * bsum_j is one more pair of small MFMAs over the 16 per-16 block sums of Q8_K (m_j duplicated),
//     the int16 sums split into int8 planes bsum = 64 * bh + bl by mmq_prep_kernel.
//   * Q6_K: the unsigned code q in [0,63] times the signed int8 scale (16-bit signed lanes), S = 6, hi in [-128,126],
//     lo in [0,63]; the "-32" of the code is the same small MFMA:  isum = 64 H + L - 32 * sum_g sc_g * bsum16_g.
//     A lane's 16 weights of a K-step are exactly one 16-group, so the scale is a per-lane scalar.
//   Only the final f32 accumulation order over super-blocks differs from the CPU.
//
// Tile mapping (wave64, v_mfma_i32_32x32x32_i8): M = tokens (A operand from LDS), N = weight rows (B operand built in
// registers): lane = (row n = lane & 31, k-half kg = lane >> 5) holds its own row's 16 weights per K-step, so d / dmin /
// scales are per-lane scalars and weights go global -> registers with no LDS round trip.  Workgroup = 8 waves:
// RW row-waves x TW token-waves with MT token tiles of 32 per wave (MT = 4: 256 rows x 128 tokens; MT = 2: 128 x 128;
// MT = 1: 256 rows x 32 tokens).  The activation tile of one super-block (tokens x 256 int8, + block-sum planes + scales) is
// staged in LDS once per workgroup (row stride 272 B: ds_read_b128 conflict-free), the next tile's global loads are
// issued before the MFMA work of the current one, and the raw weights of the next super-block likewise.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "kernels.h"

namespace mi355 {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int A_STRIDE = 272;          // 256 codes + 16 B pad per token row
constexpr int NTHREADS = 512;

__device__ __forceinline__ i32x16 mfma_i8(i32x4 a, i32x4 b, i32x16 c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ u32x4 ldg16(const void *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }

// two int8 planes of  p = scale * code  for four codes held one per byte in `w` (codes < 64, 0 <= scale < 64 for the
// unsigned form): even / odd bytes are multiplied as 16-bit lanes of one 32-bit product (no carry: p < 2^16)
template <int S>
__device__ __forceinline__ void planes_u(uint32_t w, uint32_t sc, uint32_t &hi, uint32_t &lo) {
    constexpr uint32_t LM = ((1u << S) - 1u) * 0x00010001u;
    const uint32_t pe = (w & 0x00ff00ffu) * sc;               // products of bytes 0, 2
    const uint32_t po = ((w >> 8) & 0x00ff00ffu) * sc;        // products of bytes 1, 3
    hi = ((pe >> S) & 0x00ff00ffu) | (((po >> S) & 0x00ff00ffu) << 8);
    lo = (pe & LM) | ((po & LM) << 8);
}

typedef short i16x2 __attribute__((ext_vector_type(2)));
// signed scale (int8, replicated in both 16-bit lanes of scpk): p = sc * code as 16-bit signed lanes, hi = p >> 6 (floor), lo = p & 63
__device__ __forceinline__ void planes_s6(uint32_t w, uint32_t scpk, uint32_t &hi, uint32_t &lo) {
    const i16x2 e = __builtin_bit_cast(i16x2, w & 0x00ff00ffu), o = __builtin_bit_cast(i16x2, (w >> 8) & 0x00ff00ffu);
    const i16x2 s = __builtin_bit_cast(i16x2, scpk);
    const i16x2 pe = e * s, po = o * s;                       // v_pk_mul_lo_u16: low 16 bits = the signed product
    const i16x2 six = {6, 6};
    const uint32_t he = __builtin_bit_cast(uint32_t, pe >> six), ho = __builtin_bit_cast(uint32_t, po >> six);   // v_pk_ashrrev_i16
    const uint32_t le = __builtin_bit_cast(uint32_t, pe) & 0x003f003fu, lo_ = __builtin_bit_cast(uint32_t, po) & 0x003f003fu;
    hi = (he & 0x00ff00ffu) | ((ho & 0x00ff00ffu) << 8);
    lo = le | (lo_ << 8);
}

// the same for the signed Q6_K code (q - 32) in [-32, 31]
__device__ __forceinline__ void planes_s6m32(uint32_t w, uint32_t scpk, uint32_t &hi, uint32_t &lo) {
    const i16x2 k32 = {32, 32};
    const i16x2 e = __builtin_bit_cast(i16x2, w & 0x00ff00ffu) - k32, o = __builtin_bit_cast(i16x2, (w >> 8) & 0x00ff00ffu) - k32;
    const i16x2 s = __builtin_bit_cast(i16x2, scpk);
    const i16x2 pe = e * s, po = o * s;
    const i16x2 six = {6, 6};
    const uint32_t he = __builtin_bit_cast(uint32_t, pe >> six), ho = __builtin_bit_cast(uint32_t, po >> six);
    const uint32_t le = __builtin_bit_cast(uint32_t, pe) & 0x003f003fu, lo_ = __builtin_bit_cast(uint32_t, po) & 0x003f003fu;
    hi = (he & 0x00ff00ffu) | ((ho & 0x00ff00ffu) << 8);
    lo = le | (lo_ << 8);
}

// per-lane weight-row state of one super-block: raw bytes as loaded, then what the K-steps need
template <int TYPE> struct RowSB;

template <> struct RowSB<T_Q4_K> {
    u32x4 q0, q1, q2, q3;      // chunk c: 16 bytes = 16 low nibbles (sub-block 2c) and 16 high nibbles (2c+1) of this lane's k-half
    u32x4 h;
    __device__ __forceinline__ void load(const uint8_t *row, int nb, int sb, int kg) {
        const uint8_t *b = row + (size_t)sb * 144;
        h = ldg16(b);
        q0 = ldg16(b + 16 + 16 * kg); q1 = ldg16(b + 48 + 16 * kg); q2 = ldg16(b + 80 + 16 * kg); q3 = ldg16(b + 112 + 16 * kg);
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)(h.x & 0xffff)); }
    __device__ __forceinline__ float dmin() const { return h2f((uint16_t)(h.x >> 16)); }
    // scales bytes s0..s11 in h.y h.z h.w; j<4: sc = s[j]&63, m = s[j+4]&63; j>=4: sc = (s[j+4]&15)|((s[j-4]>>6)<<4), m = (s[j+4]>>4)|((s[j]>>6)<<4)
    __device__ __forceinline__ void scales(uint32_t &sc_lo, uint32_t &sc_hi, uint32_t &mn_lo, uint32_t &mn_hi) const {
        sc_lo = h.y & 0x3f3f3f3f; mn_lo = h.z & 0x3f3f3f3f;
        sc_hi = (h.w & 0x0f0f0f0f) | ((h.y >> 2) & 0x30303030);
        mn_hi = ((h.w >> 4) & 0x0f0f0f0f) | ((h.z >> 2) & 0x30303030);
    }
    // the raw codes of group J (one per byte): the B operand of the group-scale form (scale applied to the MFMA result)
    template <int J> __device__ __forceinline__ i32x4 codes() const {
        const u32x4 v = (J >> 1) == 0 ? q0 : (J >> 1) == 1 ? q1 : (J >> 1) == 2 ? q2 : q3;
        constexpr int sh = (J & 1) * 4;
        return i32x4{(int)((v.x >> sh) & 0x0f0f0f0f), (int)((v.y >> sh) & 0x0f0f0f0f), (int)((v.z >> sh) & 0x0f0f0f0f), (int)((v.w >> sh) & 0x0f0f0f0f)};
    }
    template <int J> __device__ __forceinline__ void bop(uint32_t sc, i32x4 &bh, i32x4 &bl) const {
        const u32x4 v = (J >> 1) == 0 ? q0 : (J >> 1) == 1 ? q1 : (J >> 1) == 2 ? q2 : q3;
        constexpr int sh = (J & 1) * 4;
        uint32_t hx, lx;
        planes_u<5>((v.x >> sh) & 0x0f0f0f0f, sc, hx, lx); bh.x = (int)hx; bl.x = (int)lx;
        planes_u<5>((v.y >> sh) & 0x0f0f0f0f, sc, hx, lx); bh.y = (int)hx; bl.y = (int)lx;
        planes_u<5>((v.z >> sh) & 0x0f0f0f0f, sc, hx, lx); bh.z = (int)hx; bl.z = (int)lx;
        planes_u<5>((v.w >> sh) & 0x0f0f0f0f, sc, hx, lx); bh.w = (int)hx; bl.w = (int)lx;
    }
};

template <> struct RowSB<T_Q5_K> {
    u32x4 q0, q1, q2, q3, qh;
    u32x4 h;
    __device__ __forceinline__ void load(const uint8_t *row, int nb, int sb, int kg) {
        const uint8_t *b = row + (size_t)sb * 176;
        h = ldg16(b);
        qh = ldg16(b + 16 + 16 * kg);
        q0 = ldg16(b + 48 + 16 * kg); q1 = ldg16(b + 80 + 16 * kg); q2 = ldg16(b + 112 + 16 * kg); q3 = ldg16(b + 144 + 16 * kg);
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)(h.x & 0xffff)); }
    __device__ __forceinline__ float dmin() const { return h2f((uint16_t)(h.x >> 16)); }
    __device__ __forceinline__ void scales(uint32_t &sc_lo, uint32_t &sc_hi, uint32_t &mn_lo, uint32_t &mn_hi) const {
        sc_lo = h.y & 0x3f3f3f3f; mn_lo = h.z & 0x3f3f3f3f;
        sc_hi = (h.w & 0x0f0f0f0f) | ((h.y >> 2) & 0x30303030);
        mn_hi = ((h.w >> 4) & 0x0f0f0f0f) | ((h.z >> 2) & 0x30303030);
    }
    template <int J> __device__ __forceinline__ i32x4 codes() const {
        const u32x4 v = (J >> 1) == 0 ? q0 : (J >> 1) == 1 ? q1 : (J >> 1) == 2 ? q2 : q3;
        constexpr int sh = (J & 1) * 4;
#define Q5C(vv, hh) (int)((((vv) >> sh) & 0x0f0f0f0f) | ((((hh) >> J) & 0x01010101u) << 4))
        return i32x4{Q5C(v.x, qh.x), Q5C(v.y, qh.y), Q5C(v.z, qh.z), Q5C(v.w, qh.w)};
#undef Q5C
    }
    template <int J, int S = 5> __device__ __forceinline__ void bop(uint32_t sc, i32x4 &bh, i32x4 &bl) const {
        const u32x4 v = (J >> 1) == 0 ? q0 : (J >> 1) == 1 ? q1 : (J >> 1) == 2 ? q2 : q3;
        constexpr int sh = (J & 1) * 4;
        uint32_t hx, lx;
#define Q5W(vv, hh) ((((vv) >> sh) & 0x0f0f0f0f) | ((((hh) >> J) & 0x01010101u) << 4))
        planes_u<S>(Q5W(v.x, qh.x), sc, hx, lx); bh.x = (int)hx; bl.x = (int)lx;
        planes_u<S>(Q5W(v.y, qh.y), sc, hx, lx); bh.y = (int)hx; bl.y = (int)lx;
        planes_u<S>(Q5W(v.z, qh.z), sc, hx, lx); bh.z = (int)hx; bl.z = (int)lx;
        planes_u<S>(Q5W(v.w, qh.w), sc, hx, lx); bh.w = (int)hx; bl.w = (int)lx;
#undef Q5W
    }
};

// Q6_K device row planes: ql | qh | scales | d.  K-step s (0..7) = half n = s>>2, quarter k = s&3: this lane's 16 weights
// l = 16kg.. of that quarter are one 16-group with scale sc[8n + 2k + kg].
template <> struct RowSB<T_Q6_K> {
    u32x4 l0, l1, l2, l3;      // ql: half 0 (l, l+32), half 1 (l, l+32)
    u32x4 h0, h1;              // qh: half 0, half 1
    u32x4 scv;                 // 16 int8 scales
    uint32_t d16;
    __device__ __forceinline__ void load(const uint8_t *row, int nb, int sb, int kg) {
        l0 = ldg16(row + (size_t)sb * 128 + 16 * kg);      l1 = ldg16(row + (size_t)sb * 128 + 32 + 16 * kg);
        l2 = ldg16(row + (size_t)sb * 128 + 64 + 16 * kg); l3 = ldg16(row + (size_t)sb * 128 + 96 + 16 * kg);
        h0 = ldg16(row + (size_t)nb * 128 + (size_t)sb * 64 + 16 * kg);
        h1 = ldg16(row + (size_t)nb * 128 + (size_t)sb * 64 + 32 + 16 * kg);
        scv = ldg16(row + (size_t)nb * 192 + (size_t)sb * 16);
        d16 = *reinterpret_cast<const uint16_t *>(row + (size_t)nb * 208 + (size_t)sb * 2);
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)d16); }
    // signed scale of 16-group g, replicated into both 16-bit lanes
    __device__ __forceinline__ uint32_t scale_pk(int g) const {
        const uint32_t w = g < 4 ? scv.x : g < 8 ? scv.y : g < 12 ? scv.z : scv.w;
        const int s = (int)(int8_t)((w >> (8 * (g & 3))) & 0xff);
        return ((uint32_t)s & 0xffffu) | ((uint32_t)s << 16);
    }
    // same with the signed code (q - 32): 64 * hi + lo = sc * (q - 32), no block-sum correction needed afterwards
    template <int S> __device__ __forceinline__ void bop_signed(uint32_t scpk, i32x4 &bh, i32x4 &bl) const {
        constexpr int n = S >> 2, k = S & 3;
        const u32x4 lv = n == 0 ? ((k & 1) ? l1 : l0) : ((k & 1) ? l3 : l2);
        const u32x4 hv = n == 0 ? h0 : h1;
        constexpr int nsh = (k >> 1) * 4, hsh = 2 * k;
        uint32_t hx, lx;
#define Q6W(lw, hw) ((((lw) >> nsh) & 0x0f0f0f0f) | ((((hw) >> hsh) & 0x03030303u) << 4))
        planes_s6m32(Q6W(lv.x, hv.x), scpk, hx, lx); bh.x = (int)hx; bl.x = (int)lx;
        planes_s6m32(Q6W(lv.y, hv.y), scpk, hx, lx); bh.y = (int)hx; bl.y = (int)lx;
        planes_s6m32(Q6W(lv.z, hv.z), scpk, hx, lx); bh.z = (int)hx; bl.z = (int)lx;
        planes_s6m32(Q6W(lv.w, hv.w), scpk, hx, lx); bh.w = (int)hx; bl.w = (int)lx;
#undef Q6W
    }
    template <int S> __device__ __forceinline__ void bop(uint32_t scpk, i32x4 &bh, i32x4 &bl) const {
        constexpr int n = S >> 2, k = S & 3;
        const u32x4 lv = n == 0 ? ((k & 1) ? l1 : l0) : ((k & 1) ? l3 : l2);
        const u32x4 hv = n == 0 ? h0 : h1;
        constexpr int nsh = (k >> 1) * 4, hsh = 2 * k;
        uint32_t hx, lx;
#define Q6W(lw, hw) ((((lw) >> nsh) & 0x0f0f0f0f) | ((((hw) >> hsh) & 0x03030303u) << 4))
        planes_s6(Q6W(lv.x, hv.x), scpk, hx, lx); bh.x = (int)hx; bl.x = (int)lx;
        planes_s6(Q6W(lv.y, hv.y), scpk, hx, lx); bh.y = (int)hx; bl.y = (int)lx;
        planes_s6(Q6W(lv.z, hv.z), scpk, hx, lx); bh.z = (int)hx; bl.z = (int)lx;
        planes_s6(Q6W(lv.w, hv.w), scpk, hx, lx); bh.w = (int)hx; bl.w = (int)lx;
#undef Q6W
    }
};

// MT token tiles of 32 per wave; TW token-waves x RW row-waves = 8 waves
template <int MT> struct Geo {
    static constexpr int TW = MT == 2 ? 2 : 1, RW = 8 / TW;
    static constexpr int TOK_TILE = 32 * MT * TW, ROW_TILE = 32 * RW;
    static constexpr int LDS_A = TOK_TILE * A_STRIDE, LDS_P = TOK_TILE * 16;
    static constexpr int LDS_BYTES = LDS_A + 2 * LDS_P + TOK_TILE * 4;
    static constexpr int NST = (TOK_TILE * 16 + NTHREADS - 1) / NTHREADS;       // 16-byte staging pieces per thread
};

template <int TYPE, int MT>
__global__ __launch_bounds__(NTHREADS) void mmq_kernel(const uint8_t *W, size_t row_bytes, int n_rows, int K, int T, int n_row_tiles, int n_tok_tiles,
                                                       const int8_t *aq, const float *ad, const int8_t *abh, const int8_t *abl,
                                                       float *out, int ld_out, const float *resid) {
    using G = Geo<MT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int8_t *s_aq = reinterpret_cast<int8_t *>(smem);
    int8_t *s_bh = s_aq + G::LDS_A, *s_bl = s_bh + G::LDS_P;
    float *s_yd = reinterpret_cast<float *>(s_bl + G::LDS_P);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = K >> 8;
    // XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs; the token tiles of one row tile run on ONE
    // XCD back to back, so its weights are fetched from HBM once and re-read from that XCD's L2
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int tok_tile = loc % n_tok_tiles;
    const int row_tile = (loc / n_tok_tiles) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;                       // workgroup-uniform
    const int rw = wave % G::RW, tw = wave / G::RW;
    const int row0 = row_tile * G::ROW_TILE + rw * 32;
    const int tok0 = tok_tile * G::TOK_TILE;
    const int n = lane & 31, kg = lane >> 5;
    int my_row = row0 + n;
    const bool row_ok = my_row < n_rows;
    if (!row_ok) my_row = n_rows - 1;
    const uint8_t *rowp = W + (size_t)my_row * row_bytes;

    // staging roles: piece p = tid + NTHREADS * i -> token p / 16, 16-byte column p % 16; tokens past T re-read token T-1
    unsigned st_g[G::NST], st_l[G::NST];
#pragma unroll
    for (int i = 0; i < G::NST; i++) {
        const int p = tid + NTHREADS * i;
        int tk = p >> 4;
        if (tk >= G::TOK_TILE) tk = G::TOK_TILE - 1;
        int gt = tok0 + tk;
        if (gt >= T) gt = T - 1;
        st_g[i] = (unsigned)gt * (unsigned)K + (unsigned)(p & 15) * 16u;
        st_l[i] = (unsigned)tk * A_STRIDE + (unsigned)(p & 15) * 16u;
    }
    int ptok = tok0 + (tid < G::TOK_TILE ? tid : 0);
    if (ptok >= T) ptok = T - 1;
    const unsigned pl_g = (unsigned)ptok * (unsigned)nb;      // per-token plane / scale index base (x 16 bytes for planes)

    float facc[MT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) facc[t][r] = 0.0f;

    // ---- prologue: tile 0 into LDS, raw weights of super-block 0 into registers
    RowSB<TYPE> R;
    R.load(rowp, nb, 0, kg);
    {
        u32x4 tmp[G::NST];
#pragma unroll
        for (int i = 0; i < G::NST; i++) tmp[i] = ldg16(aq + st_g[i]);
#pragma unroll
        for (int i = 0; i < G::NST; i++) if (tid + NTHREADS * i < G::TOK_TILE * 16) *reinterpret_cast<u32x4 *>(s_aq + st_l[i]) = tmp[i];
        if (tid < G::TOK_TILE) {
            s_yd[tid] = ad[pl_g];
            *reinterpret_cast<u32x4 *>(s_bh + tid * 16) = ldg16(abh + (size_t)pl_g * 16);
            *reinterpret_cast<u32x4 *>(s_bl + tid * 16) = ldg16(abl + (size_t)pl_g * 16);
        }
    }
    __syncthreads();

    for (int sb = 0; sb < nb; sb++) {
        // ---- next activation tile: request now, park in registers across the MFMA work
        const bool more = sb + 1 < nb;
        const int sbn = more ? sb + 1 : sb;
        u32x4 nxt[G::NST];
#pragma unroll
        for (int i = 0; i < G::NST; i++) nxt[i] = ldg16(aq + st_g[i] + (unsigned)sbn * 256u);
        float nyd = 0.0f;
        u32x4 nbh = {0, 0, 0, 0}, nbl = {0, 0, 0, 0};
        if (tid < G::TOK_TILE) {
            nyd = ad[pl_g + (unsigned)sbn];
            nbh = ldg16(abh + ((size_t)pl_g + (unsigned)sbn) * 16);
            nbl = ldg16(abl + ((size_t)pl_g + (unsigned)sbn) * 16);
        }

        // ---- this super-block: scales, then 8 K-steps x MT tiles x {hi, lo}
        i32x16 H[MT], L[MT];
        const int8_t *abase = s_aq + (tw * MT * 32 + n) * A_STRIDE + 16 * kg;
        uint32_t sc_lo = 0, sc_hi = 0, mn_lo = 0, mn_hi = 0;
        if constexpr (TYPE != T_Q6_K) R.scales(sc_lo, sc_hi, mn_lo, mn_hi);
#define KSTEP(J)                                                                                              \
        {                                                                                                     \
            i32x4 bh, bl;                                                                                     \
            if constexpr (TYPE == T_Q6_K) R.template bop<J>(R.scale_pk(8 * (J >> 2) + 2 * (J & 3) + kg), bh, bl); \
            else R.template bop<J>(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff, bh, bl);                \
            _Pragma("unroll") for (int t = 0; t < MT; t++) {                                                  \
                const i32x4 a = *reinterpret_cast<const i32x4 *>(abase + t * 32 * A_STRIDE + 32 * J);          \
                if (J == 0) {                                                                                 \
                    i32x16 z;                                                                                 \
                    _Pragma("unroll") for (int r = 0; r < 16; r++) z[r] = 0;                                  \
                    H[t] = mfma_i8(a, bh, z); L[t] = mfma_i8(a, bl, z);                                       \
                } else { H[t] = mfma_i8(a, bh, H[t]); L[t] = mfma_i8(a, bl, L[t]); }                          \
            }                                                                                                 \
            __builtin_amdgcn_sched_barrier(0);   /* one K-step's operands live at a time (register pressure) */ \
        }
        KSTEP(0) KSTEP(1) KSTEP(2) KSTEP(3) KSTEP(4) KSTEP(5) KSTEP(6) KSTEP(7)
#undef KSTEP
        // ---- block-sum term: 16 per-16 sums x (mins duplicated | scales); K = 16 of 32 used (lanes kg == 0)
        i32x4 bm = {0, 0, 0, 0};
        if (kg == 0) {
            if constexpr (TYPE == T_Q6_K) { bm.x = (int)R.scv.x; bm.y = (int)R.scv.y; bm.z = (int)R.scv.z; bm.w = (int)R.scv.w; }
            else {
                bm.x = (int)perm(0, mn_lo, 0x01010000u); bm.y = (int)perm(0, mn_lo, 0x03030202u);
                bm.z = (int)perm(0, mn_hi, 0x01010000u); bm.w = (int)perm(0, mn_hi, 0x03030202u);
            }
        }
        const float dd = R.d();
        float dm = 0.0f;
        if constexpr (TYPE != T_Q6_K) dm = R.dmin();
        // raw weights of the next super-block (R is dead from here on)
        if (more) R.load(rowp, nb, sb + 1, kg);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int tl = (tw * MT + t) * 32;
            i32x4 ah = {0, 0, 0, 0}, al = {0, 0, 0, 0};
            if (kg == 0) {
                ah = *reinterpret_cast<const i32x4 *>(s_bh + (tl + n) * 16);
                al = *reinterpret_cast<const i32x4 *>(s_bl + (tl + n) * 16);
            }
            i32x16 z;
#pragma unroll
            for (int r = 0; r < 16; r++) z[r] = 0;
            __builtin_amdgcn_sched_barrier(0);
            const i32x16 mh = mfma_i8(ah, bm, z), ml = mfma_i8(al, bm, z);
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const f32x4 yd4 = *reinterpret_cast<const f32x4 *>(s_yd + tl + 8 * rq + 4 * kg);   // tokens m = 8 rq + 4 kg + (0..3)
#pragma unroll
                for (int ri = 0; ri < 4; ri++) {
                    const int r = rq * 4 + ri;
                    const float yd = yd4[ri];
                    const int bsum = 64 * mh[r] + ml[r];
                    if constexpr (TYPE == T_Q6_K) {
                        const int isum = 64 * H[t][r] + L[t][r] - 32 * bsum;
                        facc[t][r] += (dd * yd) * (float)isum;
                    } else {
                        const int isum = 32 * H[t][r] + L[t][r];
                        facc[t][r] += (dd * yd) * (float)isum - (dm * yd) * (float)bsum;
                    }
                }
            }
        }
        // ---- swap in the next tile
        __syncthreads();                             // every wave is done reading this tile
        if (more) {
#pragma unroll
            for (int i = 0; i < G::NST; i++) if (tid + NTHREADS * i < G::TOK_TILE * 16) *reinterpret_cast<u32x4 *>(s_aq + st_l[i]) = nxt[i];
            if (tid < G::TOK_TILE) {
                s_yd[tid] = nyd;
                *reinterpret_cast<u32x4 *>(s_bh + tid * 16) = nbh;
                *reinterpret_cast<u32x4 *>(s_bl + tid * 16) = nbl;
            }
        }
        __syncthreads();
    }
    // store: lane = weight row n, regs = tokens; 32 consecutive rows per token -> 128-B coalesced
    if (row_ok) {
#pragma unroll
        for (int t = 0; t < MT; t++) {
            float rv[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = (r & 3) + 8 * (r >> 2) + 4 * kg;
                int gt = tok0 + (tw * MT + t) * 32 + m;
                if (gt >= T) gt = T - 1;
                rv[r] = resid ? resid[(size_t)gt * ld_out + row0 + n] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = (r & 3) + 8 * (r >> 2) + 4 * kg;
                const int gt = tok0 + (tw * MT + t) * 32 + m;
                if (gt < T) out[(size_t)gt * ld_out + row0 + n] = rv[r] + facc[t][r];
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------------------------
// Small token counts (continuous-batching decode steps, 8 <= T <= 64): the contraction is HBM-bound again, so the
// weights are read in their GGUF form (0.56 B / weight, expanded in registers — at 32 tokens that VALU work runs at about
// the HBM rate) and the parallelism comes from K instead of tokens: workgroup = 32 weight rows x (32 * MT tokens), its 8
// waves take the super-blocks round-robin, each wave stages its OWN activation tile (no workgroup barrier in the loop),
// and the eight partial f32 tiles are summed through LDS in fixed wave order (deterministic).
// One launch covers up to three tensors that share the activation (Q / K / V), or the gate / up pair with the SwiGLU
// applied in the epilogue (both rows of a pair are contracted against the same staged tile).
struct KSplitArgs {
    MMQSeg seg[3];
    int n_seg, K, T, swiglu;
    const int8_t *aq; const float *ad; const int8_t *abh, *abl;
};

// one super-block of one 32-row tile against the wave's staged activation tile: facc += fold(H, L, block sums)
template <int TYPE, int MT>
__device__ __forceinline__ void ksplit_superblock(const RowSB<TYPE> &R, const int8_t *s_aq, const int8_t *s_bh, const int8_t *s_bl, const float *s_yd,
                                                  int n, int kg, float (&facc)[MT][16]) {
    i32x16 H[MT], L[MT];
    const int8_t *abase = s_aq + n * A_STRIDE + 16 * kg;
    uint32_t sc_lo = 0, sc_hi = 0, mn_lo = 0, mn_hi = 0;
    if constexpr (TYPE != T_Q6_K) R.scales(sc_lo, sc_hi, mn_lo, mn_hi);
#define KSTEP(J)                                                                                              \
    {                                                                                                         \
        i32x4 bh, bl;                                                                                         \
        if constexpr (TYPE == T_Q6_K) R.template bop_signed<J>(R.scale_pk(8 * (J >> 2) + 2 * (J & 3) + kg), bh, bl); \
        else R.template bop<J>(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff, bh, bl);                    \
        _Pragma("unroll") for (int t = 0; t < MT; t++) {                                                      \
            const i32x4 a = *reinterpret_cast<const i32x4 *>(abase + t * 32 * A_STRIDE + 32 * J);              \
            if (J == 0) {                                                                                     \
                i32x16 z;                                                                                     \
                _Pragma("unroll") for (int r = 0; r < 16; r++) z[r] = 0;                                      \
                H[t] = mfma_i8(a, bh, z); L[t] = mfma_i8(a, bl, z);                                           \
            } else { H[t] = mfma_i8(a, bh, H[t]); L[t] = mfma_i8(a, bl, L[t]); }                              \
        }                                                                                                     \
    }
    KSTEP(0) KSTEP(1) KSTEP(2) KSTEP(3) KSTEP(4) KSTEP(5) KSTEP(6) KSTEP(7)
#undef KSTEP
    const float dd = R.d();
    float dm = 0.0f;
    i32x4 bm = {0, 0, 0, 0};
    if constexpr (TYPE != T_Q6_K) {
        dm = R.dmin();
        if (kg == 0) {
            bm.x = (int)perm(0, mn_lo, 0x01010000u); bm.y = (int)perm(0, mn_lo, 0x03030202u);
            bm.z = (int)perm(0, mn_hi, 0x01010000u); bm.w = (int)perm(0, mn_hi, 0x03030202u);
        }
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
        i32x16 ms;
        if constexpr (TYPE != T_Q6_K) {
            i32x4 ah = {0, 0, 0, 0}, al = {0, 0, 0, 0};
            if (kg == 0) {
                ah = *reinterpret_cast<const i32x4 *>(s_bh + (t * 32 + n) * 16);
                al = *reinterpret_cast<const i32x4 *>(s_bl + (t * 32 + n) * 16);
            }
            i32x16 z;
#pragma unroll
            for (int r = 0; r < 16; r++) z[r] = 0;
            ms = mfma_i8(ah, bm, z);
#pragma unroll
            for (int r = 0; r < 16; r++) ms[r] <<= 6;
            ms = mfma_i8(al, bm, ms);
        }
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
            const f32x4 yd4 = *reinterpret_cast<const f32x4 *>(s_yd + t * 32 + 8 * rq + 4 * kg);
#pragma unroll
            for (int ri = 0; ri < 4; ri++) {
                const int r = rq * 4 + ri;
                const float yd = yd4[ri];
                if constexpr (TYPE == T_Q6_K) {
                    const int isum = 64 * H[t][r] + L[t][r];
                    facc[t][r] += (dd * yd) * (float)isum;
                } else {
                    const int isum = 32 * H[t][r] + L[t][r];
                    facc[t][r] += (dd * yd) * (float)isum - (dm * yd) * (float)ms[r];
                }
            }
        }
    }
}

// The same super-block for one token tile (T <= 32) in the GROUP-SCALE form: a K-step of the MFMA is exactly one 32-weight group of Q4_K /
// Q5_K, so the raw 4- / 5-bit codes go in as the B operand (two VALU instructions per 8 weights instead of ~10 for the two scaled planes),
// ONE MFMA per K-step yields sum_k q_k a_k of the group, and the 6-bit group scale is applied to the 16 results per lane with one
// v_mad_i32_i24 each.  With a single token tile the expansion per weight dominated the planes form (4 VALU cycles per MFMA cycle); this
// form trades the second MFMA chain for 16 multiply-adds.  The integer isum is the same number, so everything downstream is unchanged.
template <int TYPE>
__device__ __forceinline__ void ksplit_superblock_gs(const RowSB<TYPE> &R, const int8_t *s_aq, const int8_t *s_bh, const int8_t *s_bl, const float *s_yd,
                                                     int n, int kg, float (&facc)[1][16]) {
    const int8_t *abase = s_aq + n * A_STRIDE + 16 * kg;
    uint32_t sc_lo = 0, sc_hi = 0, mn_lo = 0, mn_hi = 0;
    R.scales(sc_lo, sc_hi, mn_lo, mn_hi);
    int isum[16];
#pragma unroll
    for (int r = 0; r < 16; r++) isum[r] = 0;
    i32x16 z;
#pragma unroll
    for (int r = 0; r < 16; r++) z[r] = 0;
#define GSTEP(J)                                                                                              \
    {                                                                                                         \
        const i32x16 I = mfma_i8(*reinterpret_cast<const i32x4 *>(abase + 32 * J), R.template codes<J>(), z); \
        const int sc = (int)(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff);                              \
        _Pragma("unroll") for (int r = 0; r < 16; r++) { isum[r] = __mul24(I[r], sc) + isum[r]; asm volatile("" : "+v"(isum[r])); } \
        __builtin_amdgcn_sched_barrier(0);   /* (LLVM reassociates the eight-term integer sums otherwise: all eight MFMA results live, 217 registers) */ \
    }
    GSTEP(0) GSTEP(1) GSTEP(2) GSTEP(3) GSTEP(4) GSTEP(5) GSTEP(6) GSTEP(7)
#undef GSTEP
    const float dd = R.d(), dm = R.dmin();
    i32x4 bm = {0, 0, 0, 0};
    if (kg == 0) {
        bm.x = (int)perm(0, mn_lo, 0x01010000u); bm.y = (int)perm(0, mn_lo, 0x03030202u);
        bm.z = (int)perm(0, mn_hi, 0x01010000u); bm.w = (int)perm(0, mn_hi, 0x03030202u);
    }
    i32x4 ah = {0, 0, 0, 0}, al = {0, 0, 0, 0};
    if (kg == 0) {
        ah = *reinterpret_cast<const i32x4 *>(s_bh + n * 16);
        al = *reinterpret_cast<const i32x4 *>(s_bl + n * 16);
    }
    i32x16 ms = mfma_i8(ah, bm, z);
#pragma unroll
    for (int r = 0; r < 16; r++) ms[r] <<= 6;
    ms = mfma_i8(al, bm, ms);
#pragma unroll
    for (int rq = 0; rq < 4; rq++) {
        const f32x4 yd4 = *reinterpret_cast<const f32x4 *>(s_yd + 8 * rq + 4 * kg);
#pragma unroll
        for (int ri = 0; ri < 4; ri++) {
            const int r = rq * 4 + ri;
            const float yd = yd4[ri];
            facc[0][r] += (dd * yd) * (float)isum[r] - (dm * yd) * (float)ms[r];
        }
    }
}

template <int TYPE, int MT, bool SWIGLU>
__device__ __forceinline__ void ksplit_body(const KSplitArgs &a, const MMQSeg &sg, int row_tile, uint8_t *smem) {
    constexpr int TOK = 32 * MT;
    constexpr int W_A = TOK * A_STRIDE, W_P = TOK * 16;
    constexpr int W_BYTES = W_A + 2 * W_P + TOK * 4;            // per-wave LDS region
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int8_t *s_aq = reinterpret_cast<int8_t *>(smem + wave * W_BYTES);
    int8_t *s_bh = s_aq + W_A, *s_bl = s_bh + W_P;
    float *s_yd = reinterpret_cast<float *>(s_bl + W_P);
    const int K = a.K, T = a.T, nb = K >> 8;
    const int row0 = row_tile * 32, tok0 = blockIdx.y * TOK;
    const int n = lane & 31, kg = lane >> 5;
    int my_row = row0 + n;
    if (my_row >= sg.n_rows) my_row = sg.n_rows - 1;
    const uint8_t *rowp = sg.W + (size_t)my_row * sg.row_bytes;
    const uint8_t *rowp2 = SWIGLU ? a.seg[1].W + (size_t)my_row * a.seg[1].row_bytes : nullptr;

    constexpr int NST = TOK * 16 / 64;
    int ptok = tok0 + (lane < TOK ? lane : 0);
    if (ptok >= T) ptok = T - 1;
    const unsigned pl_g = (unsigned)ptok * (unsigned)nb;

    float facc[MT][16], facc2[MT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) { facc[t][r] = 0.0f; if (SWIGLU) facc2[t][r] = 0.0f; }

    for (int sb = wave; sb < nb; sb += 8) {
        RowSB<TYPE> R;
        R.load(rowp, nb, sb, kg);
        {   // this wave's activation tile of super-block sb
            u32x4 tmp[NST];
#pragma unroll
            for (int i = 0; i < NST; i++) {
                const int p = lane + 64 * i;
                int gt = tok0 + (p >> 4);
                if (gt >= T) gt = T - 1;
                tmp[i] = ldg16(a.aq + (size_t)gt * K + (size_t)sb * 256 + (p & 15) * 16);
            }
            float yd = 0.0f;
            u32x4 vbh = {0, 0, 0, 0}, vbl = {0, 0, 0, 0};
            if (lane < TOK) {
                yd = a.ad[pl_g + (unsigned)sb];
                if (TYPE != T_Q6_K) {
                    vbh = ldg16(a.abh + ((size_t)pl_g + (unsigned)sb) * 16);
                    vbl = ldg16(a.abl + ((size_t)pl_g + (unsigned)sb) * 16);
                }
            }
            __builtin_amdgcn_wave_barrier();                    // the previous tile's reads are done (in-order LDS per wave)
#pragma unroll
            for (int i = 0; i < NST; i++) {
                const int p = lane + 64 * i;
                *reinterpret_cast<u32x4 *>(s_aq + (p >> 4) * A_STRIDE + (p & 15) * 16) = tmp[i];
            }
            if (lane < TOK) {
                s_yd[lane] = yd;
                if (TYPE != T_Q6_K) {
                    *reinterpret_cast<u32x4 *>(s_bh + lane * 16) = vbh;
                    *reinterpret_cast<u32x4 *>(s_bl + lane * 16) = vbl;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
#ifndef MI355_KSPLIT_TWO_PLANES                                  // (tools: the two-plane form for one token tile too, for comparison)
        constexpr bool GS_FORM = MT == 1 && TYPE != T_Q6_K;   // (Q6_K: 16-weight groups, a K-step spans two)
#else
        constexpr bool GS_FORM = false;
#endif
        if constexpr (GS_FORM) ksplit_superblock_gs<TYPE>(R, s_aq, s_bh, s_bl, s_yd, n, kg, facc);
        else ksplit_superblock<TYPE, MT>(R, s_aq, s_bh, s_bl, s_yd, n, kg, facc);
        if constexpr (SWIGLU) {                                 // the up row of the pair against the same tile
            RowSB<TYPE> R2;
            R2.load(rowp2, nb, sb, kg);
            if constexpr (GS_FORM) ksplit_superblock_gs<TYPE>(R2, s_aq, s_bh, s_bl, s_yd, n, kg, facc2);
            else ksplit_superblock<TYPE, MT>(R2, s_aq, s_bh, s_bl, s_yd, n, kg, facc2);
        }
    }
    // ---- sum the eight waves' partial tiles in wave order (deterministic), then store
    constexpr int NP = SWIGLU ? 2 : 1;
    __syncthreads();                                   // all activation tiles consumed: the LDS is reused for the partials
    float *part = reinterpret_cast<float *>(smem);     // [wave][NP][MT * 16][64]
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            part[((wave * NP + 0) * MT * 16 + t * 16 + r) * 64 + lane] = facc[t][r];
            if (SWIGLU) part[((wave * NP + 1) * MT * 16 + t * 16 + r) * 64 + lane] = facc2[t][r];
        }
    __syncthreads();
    for (int e = tid; e < MT * 16 * 64; e += NTHREADS) {
        float sum = 0.0f, sum2 = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; w++) {
            sum += part[(w * NP + 0) * MT * 16 * 64 + e];
            if (SWIGLU) sum2 += part[(w * NP + 1) * MT * 16 * 64 + e];
        }
        const int ln = e & 63, tr = e >> 6;            // tr = t * 16 + r
        const int t = tr >> 4, r = tr & 15;
        const int m = (r & 3) + 8 * (r >> 2) + 4 * (ln >> 5);
        const int gt = tok0 + t * 32 + m, row = row0 + (ln & 31);
        if (gt < T && row < sg.n_rows) {
            const size_t o = (size_t)gt * sg.ld_out + row;
            if (SWIGLU) sg.out[o] = (sum / (1.0f + expf(-sum))) * sum2;
            else sg.out[o] = sg.resid ? sg.resid[o] + sum : sum;
        }
    }
}

template <int MT, bool SWIGLU>
__global__ __launch_bounds__(NTHREADS) void mmq_ksplit_kernel(const KSplitArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int s = 0;
    if (a.n_seg > 1 && (int)blockIdx.x >= a.seg[1].tile0) s = 1;
    if (a.n_seg > 2 && (int)blockIdx.x >= a.seg[2].tile0) s = 2;
    if (SWIGLU) s = 0;
    const int row_tile = (int)blockIdx.x - a.seg[s].tile0;
    switch (a.seg[s].type) {
        case T_Q4_K: ksplit_body<T_Q4_K, MT, SWIGLU>(a, a.seg[s], row_tile, smem); break;
        case T_Q5_K: ksplit_body<T_Q5_K, MT, SWIGLU>(a, a.seg[s], row_tile, smem); break;
        case T_Q6_K: ksplit_body<T_Q6_K, MT, SWIGLU>(a, a.seg[s], row_tile, smem); break;
        default: break;
    }
}

// ------------------------------------------------------------------------------------------------------------------
// Pre-expanded weights ("planes"): the two int8 planes of every K-step are computed ONCE at model load and laid out
// exactly as the MFMA B operands are consumed, so the prefill kernel does no per-weight VALU work at all:
//   block(rt, sb) = 32 rows x one super-block:  [K-step J 0..7][plane 0 = hi, 1 = lo][lane 0..63][16 B]  (16 KB)
//                                               [row n 0..31][16 B meta: d | dmin << 16 (f16 bits), mins 0-3, mins 4-7, 0]
// 2 bytes per weight + 1/16 B meta.  Q6_K planes carry the SIGNED code (q - 32), so that type needs no block-sum term at all.  (Q4_K and Q5_K: as codes, below)
constexpr int PL_BLOCK = 8 * 2 * 1024 + 32 * 16;

__global__ __launch_bounds__(256) void mmq_expand_kernel(const uint8_t *W, size_t row_bytes, int n_rows, int nb, int n_rt, uint8_t *planes) {      // Q6_K
    const int lane = threadIdx.x & 63;
    const int idx = blockIdx.x * 4 + (threadIdx.x >> 6);     // (row tile, super-block)
    if (idx >= n_rt * nb) return;
    const int rt = idx / nb, sb = idx - rt * nb;
    const int n = lane & 31, kg = lane >> 5;
    int row = rt * 32 + n;
    if (row >= n_rows) row = n_rows - 1;
    RowSB<T_Q6_K> R;
    R.load(W + (size_t)row * row_bytes, nb, sb, kg);
    uint8_t *blk = planes + (size_t)idx * PL_BLOCK;
#define EXP(J)                                                                                                 \
    {                                                                                                          \
        i32x4 bh, bl;                                                                                          \
        R.template bop_signed<J>(R.scale_pk(8 * (J >> 2) + 2 * (J & 3) + kg), bh, bl);                         \
        *reinterpret_cast<i32x4 *>(blk + (J * 2) * 1024 + lane * 16) = bh;                                     \
        *reinterpret_cast<i32x4 *>(blk + (J * 2 + 1) * 1024 + lane * 16) = bl;                                 \
    }
    EXP(0) EXP(1) EXP(2) EXP(3) EXP(4) EXP(5) EXP(6) EXP(7)
#undef EXP
    if (kg == 0) *reinterpret_cast<u32x4 *>(blk + 16384 + n * 16) = u32x4{R.d16, 0, 0, 0};
}

// Q2_K and Q3_K into the same plane format (their prompts then run on the kernels below; there is no expand-on-the-fly form for them):
//   Q2_K: p = scale * code <= 15 * 3, planes as Q4_K's (hi = p >> 5, lo = p & 31); sub-block 2 J + kg (16 weights) is exactly a lane's share of K-step J;
//         its sixteen 4-bit mins go into the meta words as nibbles (y: sub-blocks 0-7, z: 8-15) and w = 1 tells the fold to read them that way
//         (one min per block sum instead of one per two);
//   Q3_K: p = (scale - 32) * code with code in [-4, 3]: signed, 16-weight groups, no mins - planes as Q6_K's (hi = p >> 6 floored, lo = p & 63).
// device rows (dev_common.h): Q2_K [qs nb*64][scales nb*16][d, dmin nb*4];  Q3_K [hmask nb*32][qs nb*64][scales nb*12][d nb*2]
template <int TYPE>
__global__ __launch_bounds__(256) void mmq_expand_small_kernel(const uint8_t *W, size_t row_bytes, int n_rows, int nb, int n_rt, uint8_t *planes) {
    const int lane = threadIdx.x & 63;
    const int idx = blockIdx.x * 4 + (threadIdx.x >> 6);     // (row tile, super-block)
    if (idx >= n_rt * nb) return;
    const int rt = idx / nb, sb = idx - rt * nb;
    const int n = lane & 31, kg = lane >> 5;
    int row = rt * 32 + n;
    if (row >= n_rows) row = n_rows - 1;
    const uint8_t *r = W + (size_t)row * row_bytes;
    uint8_t *blk = planes + (size_t)idx * PL_BLOCK;
    const size_t qs_off = TYPE == T_Q2_K ? 0 : (size_t)nb * 32;
    // this lane's code bytes: l = 16 kg .. 16 kg + 15 of both 32-byte halves
    const u32x4 q0 = ldg16(r + qs_off + (size_t)sb * 64 + 16 * kg), q1 = ldg16(r + qs_off + (size_t)sb * 64 + 32 + 16 * kg);
    u32x4 hm = {0, 0, 0, 0};
    int sc[16];
    uint32_t mn_lo = 0, mn_hi = 0;
    if (TYPE == T_Q2_K) {
        const uint8_t *scp = r + (size_t)nb * 64 + (size_t)sb * 16;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int b = scp[i];
            sc[i] = b & 15;
            if (i < 8) mn_lo |= (uint32_t)(b >> 4) << (4 * i); else mn_hi |= (uint32_t)(b >> 4) << (4 * (i - 8));
        }
    } else {
        hm = ldg16(r + (size_t)sb * 32 + 16 * kg);
        const uint8_t *scp = r + (size_t)nb * 96 + (size_t)sb * 12;
#pragma unroll
        for (int i = 0; i < 16; i++) {   // 6-bit scale i: low 4 bits = nibble i of bytes 0-7 (low nibbles 0-7, high nibbles 8-15), high 2 bits = bit pair i / 4 of byte 8 + i % 4
            const int low = i < 8 ? (scp[i] & 15) : (scp[i - 8] >> 4);
            sc[i] = (low | (((scp[8 + (i & 3)] >> (2 * (i >> 2))) & 3) << 4)) - 32;
        }
    }
#pragma unroll
    for (int J = 0; J < 8; J++) {
        const u32x4 qv = (J >> 2) ? q1 : q0;
        const int sh = 2 * (J & 3);
        const int s = sc[2 * J + kg];
        const uint32_t cw[4] = {(qv.x >> sh) & 0x03030303u, (qv.y >> sh) & 0x03030303u, (qv.z >> sh) & 0x03030303u, (qv.w >> sh) & 0x03030303u};
        const uint32_t hw[4] = {hm.x, hm.y, hm.z, hm.w};
        uint32_t hv[4], lv[4];
#pragma unroll
        for (int w = 0; w < 4; w++) {
            uint32_t hx = 0, lx = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                int code = (int)((cw[w] >> (8 * b)) & 3u);
                int p;
                if (TYPE == T_Q2_K) { p = s * code; hx |= (uint32_t)((p >> 5) & 0xff) << (8 * b); lx |= (uint32_t)(p & 31) << (8 * b); }
                else {
                    if (!((hw[w] >> (8 * b + J)) & 1u)) code -= 4;          // bit J = 4 (J >> 2) + (J & 3) of the element's hmask byte
                    p = s * code;
                    hx |= (uint32_t)((p >> 6) & 0xff) << (8 * b); lx |= (uint32_t)(p & 63) << (8 * b);
                }
            }
            hv[w] = hx; lv[w] = lx;
        }
        *reinterpret_cast<u32x4 *>(blk + (J * 2) * 1024 + lane * 16) = u32x4{hv[0], hv[1], hv[2], hv[3]};
        *reinterpret_cast<u32x4 *>(blk + (J * 2 + 1) * 1024 + lane * 16) = u32x4{lv[0], lv[1], lv[2], lv[3]};
    }
    if (kg == 0) {
        u32x4 m = {0, 0, 0, 0};
        if (TYPE == T_Q2_K) { m.x = *reinterpret_cast<const uint32_t *>(r + (size_t)nb * 80 + (size_t)sb * 4); m.y = mn_lo; m.z = mn_hi; m.w = 1u; }
        else m.x = *reinterpret_cast<const uint16_t *>(r + (size_t)nb * 108 + (size_t)sb * 2);
        *reinterpret_cast<u32x4 *>(blk + 16384 + n * 16) = m;
    }
}
// Q4_K as codes, the kernels make the planes of them a super-block ahead: a scale is 8 s1 + s0, and a code times three bits stays in its byte, so one 16-bit multiplication makes two
// products:  isum = 8 (s1 q . a) + (s0 q . a).  Q5_K with the seven low bits of p as one plane and the four high ones as nibbles of two K-steps:  isum = 128 (hi . a) + (lo . a).
//   block(rt, sb) = 32 rows x one super-block:  Q4_K [codes of K-steps 2 c and 2 c + 1, a nibble each: c 0..3][lane][16 B]      [row n][16 B: s0, s1 of the eight groups]
//                                               Q5_K [low plane of K-step 0..7][lane][16 B][high nibbles of K-steps 2 c, 2 c + 1][lane][16 B]
//                                               [row n][16 B meta as above]
enum PlaneForm { PF_SIGNED, PF_MINS, PF_CODES, PF_NIBBLES };
__host__ __device__ constexpr PlaneForm plane_form(int type) { return type == T_Q4_K ? PF_CODES : type == T_Q5_K ? PF_NIBBLES : type == T_Q2_K ? PF_MINS : PF_SIGNED; }
__host__ __device__ constexpr int plane_words(int form) { return form == PF_CODES ? 4096 : form == PF_NIBBLES ? 12288 : 16384; }        // bytes of a block in front of its rows' words
__host__ __device__ constexpr int plane_block(int form) { return plane_words(form) + (form == PF_CODES ? 1024 : 512); }
__host__ __device__ constexpr int plane_shift(int form) { return form == PF_SIGNED ? 6 : form == PF_MINS ? 5 : form == PF_NIBBLES ? 7 : 3; }
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
// K-step J of what a lane holds of a block: codes, its 16 B of them and the scales of K-steps 2 (J / 2) and + 1 -> both planes; nibbles -> the high one
template <int FORM, int J>
__device__ __forceinline__ void expand_words(u32x4 raw, uint32_t sw, i32x4 &hi, i32x4 &lo) {
    const u16x2 s = __builtin_bit_cast(u16x2, perm(0, sw, J & 1 ? 0x0c030c02u : 0x0c010c00u)), s0 = {s.x, s.x}, s1 = {s.y, s.y};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t q = (J & 1 ? raw[e] >> 4 : raw[e]) & 0x0f0f0f0fu;
        if (FORM == PF_NIBBLES) { hi[e] = (int)q; continue; }
        hi[e] = (int)__builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, q) * s1));
        lo[e] = (int)__builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, q) * s0));
    }
}
template <int TYPE>
__global__ __launch_bounds__(256) void mmq_pack_kernel(const uint8_t *W, size_t row_bytes, int n_rows, int nb, int n_rt, uint8_t *planes) {
    constexpr int FORM = plane_form(TYPE), WORDS = plane_words(FORM), BLOCK = plane_block(FORM);
    const int lane = threadIdx.x & 63;
    const int idx = blockIdx.x * 4 + (threadIdx.x >> 6);     // (row tile, super-block)
    if (idx >= n_rt * nb) return;
    const int rt = idx / nb, sb = idx - rt * nb;
    const int n = lane & 31, kg = lane >> 5;
    int row = rt * 32 + n;
    if (row >= n_rows) row = n_rows - 1;
    RowSB<TYPE> R;
    R.load(W + (size_t)row * row_bytes, nb, sb, kg);
    uint8_t *blk = planes + (size_t)idx * BLOCK;
    u32x4 *o = reinterpret_cast<u32x4 *>(blk) + lane;
    uint32_t sc_lo, sc_hi, mn_lo, mn_hi;
    R.scales(sc_lo, sc_hi, mn_lo, mn_hi);
    if constexpr (FORM == PF_CODES) {
        o[0] = R.q0; o[64] = R.q1; o[128] = R.q2; o[192] = R.q3;
        u32x4 v;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t w = (c < 2 ? sc_lo : sc_hi) >> (16 * (c & 1)), a = w & 0xff, b = (w >> 8) & 0xff;
            v[c] = (a & 7) | (a >> 3) << 8 | (b & 7) << 16 | (b >> 3) << 24;
        }
        if (kg) *reinterpret_cast<u32x4 *>(blk + WORDS + n * 16) = v;
    } else {
        u32x4 hi;                                               // of a pair of K-steps
#define OUT(J)                                                                                                 \
        {                                                                                                      \
            i32x4 h, l;                                                                                        \
            R.template bop<J, 7>(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff, h, l);                     \
            o[64 * J] = __builtin_bit_cast(u32x4, l);                                                          \
            _Pragma("unroll") for (int e = 0; e < 4; e++) hi[e] = J & 1 ? hi[e] | (uint32_t)h[e] << 4 : (uint32_t)h[e]; \
            if (J & 1) o[64 * (8 + J / 2)] = hi;                                                               \
        }
        OUT(0) OUT(1) OUT(2) OUT(3) OUT(4) OUT(5) OUT(6) OUT(7)
#undef OUT
    }
    if (kg == 0) *reinterpret_cast<u32x4 *>(blk + BLOCK - 512 + n * 16) = u32x4{R.h.x, mn_lo, mn_hi, 0};
}

// Several tensors that share the activation and whose plane sets lie back to back in memory (attn_q | attn_k | attn_v) run as
// ONE launch over the concatenated rows: rows [row_end[s-1], row_end[s]) go to out[s] with leading dimension ld[s] (segment
// boundaries are multiples of 32, so a wave's 32-row tile belongs to one segment).  A 1024-row tensor alone fills a quarter of
// the chip and takes as long as a 4096-row one (34 vs 38 us at 512 tokens); the three together take 59 us instead of 106.
struct PlanesOut {
    float *out[3];
    int ld[3];
    int row_end[3];
    int n_seg;
    int form[3];            // PlaneForm of a segment, and where its blocks begin: mmq_planes2_kernel<P2_MIXED> only
    size_t at[3];
};

template <int FORM, int MT>
__global__ __launch_bounds__(NTHREADS) void mmq_planes_kernel(const uint8_t *planes, int n_rows, int K, int T, int n_row_tiles, int n_tok_tiles,
                                                              const int8_t *aq, const float *ad, const int8_t *abh, const int8_t *abl,
                                                              const PlanesOut po, const float *resid) {
    using G = Geo<MT>;
    constexpr bool MINS = FORM != PF_SIGNED, PACKED = FORM >= PF_CODES;
    constexpr int SH = plane_shift(FORM), BLOCK = plane_block(FORM), WORDS = plane_words(FORM);
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    // two activation tiles: super-block sb is read from buffer sb & 1 while sb + 1 is written into the other one, so one
    // barrier per super-block suffices and the LDS writes overlap the other waves' MFMA work
    uint8_t *buf0 = smem, *buf1 = smem + G::LDS_BYTES;
    auto p_aq = [&](int b) { return reinterpret_cast<int8_t *>(b ? buf1 : buf0); };
    auto p_bh = [&](int b) { return p_aq(b) + G::LDS_A; };
    auto p_bl = [&](int b) { return p_aq(b) + G::LDS_A + G::LDS_P; };
    auto p_yd = [&](int b) { return reinterpret_cast<float *>(p_aq(b) + G::LDS_A + 2 * G::LDS_P); };
    int8_t *s_aq = p_aq(0), *s_bh = p_bh(0), *s_bl = p_bl(0);
    float *s_yd = p_yd(0);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = K >> 8;
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int tok_tile = loc % n_tok_tiles;
    const int row_tile = (loc / n_tok_tiles) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;                       // workgroup-uniform
    const int rw = wave % G::RW, tw = wave / G::RW;
    const int rt32 = row_tile * G::RW + rw;                    // 32-row tile of this wave
    const int n_rt32 = (n_rows + 31) >> 5;
    const int row0 = rt32 * 32;
    const int tok0 = tok_tile * G::TOK_TILE;
    const int n = lane & 31, kg = lane >> 5;
    const bool tile_ok = rt32 < n_rt32;
    const uint8_t *blk0 = planes + (size_t)(tile_ok ? rt32 : n_rt32 - 1) * nb * BLOCK;
    const unsigned b_off = (unsigned)lane * 16u;

    unsigned st_g[G::NST], st_l[G::NST];
#pragma unroll
    for (int i = 0; i < G::NST; i++) {
        const int p = tid + NTHREADS * i;
        int tk = p >> 4;
        if (tk >= G::TOK_TILE) tk = G::TOK_TILE - 1;
        int gt = tok0 + tk;
        if (gt >= T) gt = T - 1;
        st_g[i] = (unsigned)gt * (unsigned)K + (unsigned)(p & 15) * 16u;
        st_l[i] = (unsigned)tk * A_STRIDE + (unsigned)(p & 15) * 16u;
    }
    int ptok = tok0 + (tid < G::TOK_TILE ? tid : 0);
    if (ptok >= T) ptok = T - 1;
    const unsigned pl_g = (unsigned)ptok * (unsigned)nb;

    float facc[MT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) facc[t][r] = 0.0f;

    // ---- prologue: B operands and meta of super-block 0 into registers, activation tile 0 into LDS
    // ring of K-steps: 4 (half a super-block ahead) where two token tiles per wave leave no registers for more; 8 (a whole
    // super-block ahead) with one tile per wave, whose 2 MFMAs per K-step otherwise cover only 256 cycles of the planes' latency
    constexpr int RING = MT == 1 ? 8 : 4;
    i32x4 Bh[RING], Bl[RING];                                   // (a slot's Bh holds codes and nibbles as they are)
    auto ld_b = [&](const uint8_t *blk, int j, int slot) {
        Bh[slot] = *reinterpret_cast<const i32x4 *>(blk + (FORM == PF_CODES ? j >> 1 : FORM == PF_NIBBLES ? 8 + (j >> 1) : 2 * j) * 1024 + b_off);
        if (FORM != PF_CODES) Bl[slot] = *reinterpret_cast<const i32x4 *>(blk + (FORM == PF_NIBBLES ? j : 2 * j + 1) * 1024 + b_off);
    };
#pragma unroll
    for (int j = 0; j < RING; j++) ld_b(blk0, j, j);
    u32x4 meta = ldg16(blk0 + BLOCK - 512 + n * 16), scales = FORM == PF_CODES ? ldg16(blk0 + WORDS + n * 16) : meta;
    {
        u32x4 tmp[G::NST];
#pragma unroll
        for (int i = 0; i < G::NST; i++) tmp[i] = ldg16(aq + st_g[i]);
#pragma unroll
        for (int i = 0; i < G::NST; i++) if (tid + NTHREADS * i < G::TOK_TILE * 16) *reinterpret_cast<u32x4 *>(s_aq + st_l[i]) = tmp[i];
        if (tid < G::TOK_TILE) {
            s_yd[tid] = ad[pl_g];
            if (MINS) {
                *reinterpret_cast<u32x4 *>(s_bh + tid * 16) = ldg16(abh + (size_t)pl_g * 16);
                *reinterpret_cast<u32x4 *>(s_bl + tid * 16) = ldg16(abl + (size_t)pl_g * 16);
            }
        }
    }
    __syncthreads();

    for (int sb = 0; sb < nb; sb++) {
        s_aq = p_aq(sb & 1); s_bh = p_bh(sb & 1); s_bl = p_bl(sb & 1); s_yd = p_yd(sb & 1);
        const bool more = sb + 1 < nb;
        const int sbn = more ? sb + 1 : sb;
        const uint8_t *blkn = blk0 + (size_t)sbn * BLOCK;
        // next activation tile: request now, park in registers across the MFMA work
        u32x4 nxt[G::NST];
#pragma unroll
        for (int i = 0; i < G::NST; i++) nxt[i] = ldg16(aq + st_g[i] + (unsigned)sbn * 256u);
        float nyd = 0.0f;
        u32x4 nbh = {0, 0, 0, 0}, nbl = {0, 0, 0, 0};
        if (tid < G::TOK_TILE) {
            nyd = ad[pl_g + (unsigned)sbn];
            if (MINS) {
                nbh = ldg16(abh + ((size_t)pl_g + (unsigned)sbn) * 16);
                nbl = ldg16(abl + ((size_t)pl_g + (unsigned)sbn) * 16);
            }
        }
        const u32x4 mcur = meta, scur = scales;
        meta = ldg16(blkn + BLOCK - 512 + n * 16);
        if (FORM == PF_CODES) scales = ldg16(blkn + WORDS + n * 16);

        i32x16 H[MT], L[MT];
        const int8_t *abase = s_aq + (tw * MT * 32 + n) * A_STRIDE + 16 * kg;
        const uint8_t *blkc = blk0 + (size_t)sb * BLOCK;
        // K-step J: MFMAs on ring slot J & 3, then the slot is refilled with the operand four K-steps ahead (same
        // super-block for J < 4, the next one otherwise): every B register waits half an iteration before its use
        // A fragments are read one K-step ahead of the MFMAs that use them (two register sets)
        i32x4 a0[MT], a1[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) a0[t] = *reinterpret_cast<const i32x4 *>(abase + t * 32 * A_STRIDE);
#define KSTEP(J, ACUR, ANXT)                                                                                  \
        {                                                                                                     \
            if (J < 7) {                                                                                      \
                _Pragma("unroll") for (int t = 0; t < MT; t++)                                                \
                    ANXT[t] = *reinterpret_cast<const i32x4 *>(abase + t * 32 * A_STRIDE + 32 * (J + 1));     \
            }                                                                                                 \
            i32x4 bh = Bh[J & (RING - 1)], bl = Bl[J & (RING - 1)];                                           \
            if constexpr (PACKED) expand_words<FORM, J>(__builtin_bit_cast(u32x4, bh), scur[J >> 1], bh, bl); \
            _Pragma("unroll") for (int t = 0; t < MT; t++) {                                                  \
                if (J == 0) {                                                                                 \
                    i32x16 z;                                                                                 \
                    _Pragma("unroll") for (int r = 0; r < 16; r++) z[r] = 0;                                  \
                    H[t] = mfma_i8(ACUR[t], bh, z); L[t] = mfma_i8(ACUR[t], bl, z);                           \
                } else { H[t] = mfma_i8(ACUR[t], bh, H[t]); L[t] = mfma_i8(ACUR[t], bl, L[t]); }              \
            }                                                                                                 \
            ld_b(RING == 8 ? blkn : J < 4 ? blkc : blkn, RING == 8 ? J : (J + 4) & 7, J & (RING - 1));         \
        }
        KSTEP(0, a0, a1) KSTEP(1, a1, a0) KSTEP(2, a0, a1) KSTEP(3, a1, a0) KSTEP(4, a0, a1) KSTEP(5, a1, a0) KSTEP(6, a0, a1) KSTEP(7, a1, a0)
#undef KSTEP
        const float dd = h2f((uint16_t)(mcur.x & 0xffff));
        float dm = 0.0f;
        i32x4 bm = {0, 0, 0, 0};
        if (MINS) {
            dm = h2f((uint16_t)(mcur.x >> 16));
            if (kg == 0) {
                if (mcur.w) {           // sixteen 4-bit mins, one per block sum (Q2_K planes): nibbles -> bytes in block-sum order
                    const uint32_t ey = mcur.y & 0x0f0f0f0fu, oy = (mcur.y >> 4) & 0x0f0f0f0fu, ez = mcur.z & 0x0f0f0f0fu, oz = (mcur.z >> 4) & 0x0f0f0f0fu;
                    bm.x = (int)perm(oy, ey, 0x05010400u); bm.y = (int)perm(oy, ey, 0x07030602u);
                    bm.z = (int)perm(oz, ez, 0x05010400u); bm.w = (int)perm(oz, ez, 0x07030602u);
                } else {
                    bm.x = (int)perm(0, mcur.y, 0x01010000u); bm.y = (int)perm(0, mcur.y, 0x03030202u);
                    bm.z = (int)perm(0, mcur.z, 0x01010000u); bm.w = (int)perm(0, mcur.z, 0x03030202u);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int tl = (tw * MT + t) * 32;
            i32x16 ms;                                // block-sum term: 64 * (bh . m) + (bl . m) in ONE accumulator
            if (MINS) {
                i32x4 ah = {0, 0, 0, 0}, al = {0, 0, 0, 0};
                if (kg == 0) {
                    ah = *reinterpret_cast<const i32x4 *>(s_bh + (tl + n) * 16);
                    al = *reinterpret_cast<const i32x4 *>(s_bl + (tl + n) * 16);
                }
                i32x16 z;
#pragma unroll
                for (int r = 0; r < 16; r++) z[r] = 0;
                ms = mfma_i8(ah, bm, z);
#pragma unroll
                for (int r = 0; r < 16; r++) ms[r] <<= 6;
                ms = mfma_i8(al, bm, ms);
            }
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const f32x4 yd4 = *reinterpret_cast<const f32x4 *>(s_yd + tl + 8 * rq + 4 * kg);
#pragma unroll
                for (int ri = 0; ri < 4; ri++) {
                    const int r = rq * 4 + ri;
                    const float yd = yd4[ri];
                    const int isum = (H[t][r] << SH) + L[t][r];
                    // yd * (d * isum - dmin * msum) with explicit fmas: 6 VALU ops per output instead of 10 (this fold was the
                    // kernel's VALU bottleneck: PMC showed 9.5 VALU instructions per MFMA); one rounding fewer than the CPU's
                    // expression, far inside the 2e-5 parity bound
                    if (MINS) {
                        const float t0 = fmaf(dd, (float)isum, -(dm * (float)ms[r]));
                        facc[t][r] = fmaf(yd, t0, facc[t][r]);
                    } else {
                        facc[t][r] = fmaf(yd * dd, (float)isum, facc[t][r]);
                    }
                }
            }
        }
        if (more) {                                  // next tile into the other buffer (nobody reads it during this iteration)
            int8_t *w_aq = p_aq((sb + 1) & 1), *w_bh = p_bh((sb + 1) & 1), *w_bl = p_bl((sb + 1) & 1);
            float *w_yd = p_yd((sb + 1) & 1);
#pragma unroll
            for (int i = 0; i < G::NST; i++) if (tid + NTHREADS * i < G::TOK_TILE * 16) *reinterpret_cast<u32x4 *>(w_aq + st_l[i]) = nxt[i];
            if (tid < G::TOK_TILE) {
                w_yd[tid] = nyd;
                if (MINS) {
                    *reinterpret_cast<u32x4 *>(w_bh + tid * 16) = nbh;
                    *reinterpret_cast<u32x4 *>(w_bl + tid * 16) = nbl;
                }
            }
        }
        __syncthreads();                             // tile sb + 1 complete; every wave is done reading tile sb
    }
    // store: lane = weight row n, regs = tokens; 32 consecutive rows per token -> 128-B coalesced.  Residual values are
    // all requested before the first add (a load + wait per element serialised the epilogue).
    if (tile_ok && row0 + n < n_rows) {
        int sg = 0;
        if (po.n_seg > 1 && row0 >= po.row_end[0]) sg = 1;
        if (po.n_seg > 2 && row0 >= po.row_end[1]) sg = 2;
        float *out = po.out[sg] - (sg ? po.row_end[sg - 1] : 0);       // so that out[t * ld + row] addresses the segment's own row
        const int ld_out = po.ld[sg];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            float rv[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = (r & 3) + 8 * (r >> 2) + 4 * kg;
                int gt = tok0 + (tw * MT + t) * 32 + m;
                if (gt >= T) gt = T - 1;
                rv[r] = resid ? resid[(size_t)gt * ld_out + row0 + n] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = (r & 3) + 8 * (r >> 2) + 4 * kg;
                const int gt = tok0 + (tw * MT + t) * 32 + m;
                if (gt < T) out[(size_t)gt * ld_out + row0 + n] = rv[r] + facc[t][r];
            }
        }
    }
}

// ---- the same contraction in 128-row x 256-token workgroup tiles: activations through LDS, weights straight into registers.
// Eight waves: wave (rw, tw) owns 32 rows x 128 tokens of the tile, i.e. the 32-row tile rw of token half tw.  Per super-block a wave has its planes as the sixteen MFMA operands that they
// are, in 64 registers, while it walks its four token tiles; both halves ask for the same words at about the same time, so the second finds them in the vector L1.  The words of the next
// super-block are asked for in the last token tile, as the operands' registers come free; of packed forms they wait in the registers of the operands that are made of them, K-step by K-step two
// steps ahead of the first token tile.  The 256 x 256 activation codes come by LDS-DMA one super-block ahead (two buffers, one barrier per super-block):
//   codes  64 KiB = [token 0..255][16 pieces of 16 B]; piece p of token t sits in slot p ^ (t & 15) (applied on the SOURCE side of the DMA, whose LDS side is
//          lane-linear), so the 16 lanes of a ds_read_b128 phase hit all 64 banks
//   block sums 8 KiB (int16, turned into f16 in place by the wave that fetched them), the rows' words (scales, d / dmin / mins), and the tokens' scales (three sets: a
//          fold reaches into the next super-block)
// The f32 fold of a token tile (five vector instructions an output) runs BETWEEN the MFMAs of the next tile, two outputs per K-step, on the other of two accumulator
// pairs: a wave in an MFMA phase of its own leaves the vector unit idle, and one in a fold of its own the matrix cores.
//
// What bounds it: gate | up of an 8B layer (14336 x 4096 twice, Q4_K, 512 tokens) is 448 workgroups, two rounds of the 256 CUs of which the second is three quarters full; in each a SIMD issues
// 2176 MFMAs of 32 cycles, so both rounds are 58 us at 2.4 GHz; but MFMAs of random operands alone run at 1.6 GHz here, with ten f32 instructions a pair of them at 1.5, of zeros at 2.4: the
// card's power.  What instructions and bytes cost comes on top of the MFMAs, whichever unit has room: of a round of 70 us (2048 tokens) the expansion of codes is 16, the fold 12, and what is
// left without both 42 (copies of the kernel without the one, the other, both); of 55 with all-zero operands the activations' way to LDS is 3.  profiles/prompt_contraction.txt.
// So bytes were taken out where instructions do not cost as much (us, before -> now, with weights from HBM): planes of 2 B a weight against Q4_K codes of 0.63 B: gate | up at 130, 256
// and 512 tokens 70 -> 49, 79 -> 61, 159 -> 153; Q5_K as 1.5 B (a byte and a nibble: 6 instructions a K-step; as codes of a byte, 17, eight layers of a 7B model at 512 tokens 3179 us, as planes 3035,
// so 2956): experts of an 8x7B layer, 611 tokens, gate | up 544 -> 455.
// Tried, and slower: two 128 x 128 workgroups per CU, each with planes of its own (192 KiB), by 4 %; 16 x 16 x 64 MFMA tiles, which read twice the registers per product, the same; touching the
// super-block after the next one, to have it in the L2 (64 lines an instruction), 12 %; the DMA's requests spread over the K-steps, 3 %; workgroups that walk equal shares of 64-token
// pairs, by 12 % at 512 tokens: the CUs that the second round leaves idle cost nothing while the others' bytes and power bound it.  One MFMA a group and the scale on its sixteen results: a fifth more.
// The block-sum ("mins") term is one v_mfma_f32_32x32x16_f16 per tile: the 16 block sums (|.| <= 2032) and the 6-bit mins are exact in f16 and their 16 products sum to
// < 2^24, so the f32 result IS the integer msum.  The integer sums, the fold and the f32 order over super-blocks are those of mmq_planes_kernel: results are bit-identical.
__device__ __forceinline__ unsigned lds_addr32(const void *p) { return (unsigned)(uintptr_t)p; }
// lane l: 16 B from gbase + voff (voff per lane) to LDS dst + 16 l
__device__ __forceinline__ void dma16_s(const void *gbase, unsigned voff, unsigned lds_dst) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff), "s"(gbase), "s"(lds_dst) : "memory");
}
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// lane l: 4 B from gbase + voff to LDS dst + 4 l
__device__ __forceinline__ void dma4_s(const void *gbase, unsigned voff, unsigned lds_dst) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff), "s"(gbase), "s"(lds_dst) : "memory");
}

constexpr int P2_ROWS = 128, P2_TOK = 256;
constexpr int P2_BS = 65536, P2_META = P2_BS + 8192, P2_BUF = P2_META + 4096, P2_YD = 2 * P2_BUF, P2_YDB = 640, P2_LDS = P2_YD + 6 * P2_YDB;

struct P2Args {
    const uint8_t *planes, *planes_up;
    int n_rows, K, T;
    const int8_t *aq; const float *ad; const int16_t *absum;
    const float *resid; float *ws; int n_split;
};
typedef const __attribute__((address_space(1))) uint8_t gbytes;
// a pointer that is the same in every lane, in scalar registers
__device__ __forceinline__ gbytes *scalar_ptr(const void *p) {
    const uint64_t v = (uint64_t)p;
    return (gbytes *)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
}
// NT: token tiles of 32; FULL: every token of the workgroup's tile exists.  SHARED: the rows' words, the same for both halves, come once, by the first (codes: two sets do not fit)
template <int FORM, int NT, bool FULL, bool SHARED>
__device__ __forceinline__ void planes2_loop(gbytes *blk0, const P2Args &a, int sb_lo, int nb, int tok0, int tid, int tw, uint8_t *smem_wg, float (&facc)[4][16]) {
    constexpr bool MINS = FORM != PF_SIGNED, PACKED = FORM >= PF_CODES;
    constexpr int SH = plane_shift(FORM), BLOCK = plane_block(FORM), WORDS = plane_words(FORM);
    // (a half's four waves stage their own tokens: `wave` is the wave's index in its half)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const int n = lane & 31, kg = lane >> 5;
    const int nb_all = a.K >> 8;
    const uint8_t *sm_bs = smem_wg + P2_BS + tw * 4096, *sm_yd = smem_wg + P2_YD + tw * P2_YDB, *sm_a = smem_wg + tw * 32768;
    const unsigned meta_at = FORM == PF_CODES ? (unsigned)wave * 1024u : (unsigned)((SHARED ? 0 : tw * 4) + wave) * 512u;
    const uint8_t *sm_meta = smem_wg + P2_META + meta_at;
    const unsigned lds0 = lds_addr32(smem_wg);
    const int last = a.T - 1 - tok0;                            // (tokens past the end read the last one; never stored)
    auto dma = [&](int sb, int buf, int y3) {                   // tokens 32 wave .. + 31 of super-block sb, and the scale words of the wave's rows
        const unsigned dst = lds0 + (unsigned)buf * P2_BUF;
        int l = lane;
        asm volatile("" : "+v"(l));                             // (the offsets are formed here, every time: hoisted out of the loop they would cost ten registers)
        if (!SHARED || tw == 0) {
            const uint8_t *mw = (const uint8_t *)scalar_ptr((const uint8_t *)blk0 + (size_t)sb * BLOCK + WORDS);
            const unsigned to = dst + P2_META + meta_at;
            if (FORM == PF_CODES) dma16_s(mw, l * 16u, to);
            else { dma4_s(mw, l * 4u, to); dma4_s(mw + 256, l * 4u, to + 256u); }
        }
        const size_t sbg = (size_t)(sb_lo + sb);
        if (NT == 4 || wave < NT) {
            const int q4 = l >> 4, p16 = l & 15;
            if (FULL) {
                const int8_t *g = (const int8_t *)scalar_ptr(a.aq + (size_t)(tok0 + 32 * wave) * a.K + sbg * 256);
                const unsigned off = (unsigned)q4 * (unsigned)a.K + (unsigned)(p16 ^ q4) * 16u;      // of the wave's first four tokens
#pragma unroll
                for (int k = 0; k < 8; k++) dma16_s(g + (size_t)(4 * k) * a.K, off ^ (64u * (k & 3)), dst + (unsigned)(32 * tw + 8 * wave + k) * 1024u);
            } else {
                const int8_t *g = (const int8_t *)scalar_ptr(a.aq + (size_t)tok0 * a.K + sbg * 256);
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const int t = 32 * wave + 4 * k + q4;
                    dma16_s(g, (unsigned)(t < last ? t : last) * (unsigned)a.K + (unsigned)(p16 ^ (4 * (k & 3) + q4)) * 16u, dst + (unsigned)(32 * tw + 8 * wave + k) * 1024u);
                }
            }
            const int bt = 32 * wave + (l >> 1), yt = 32 * wave + l;
            if (MINS) dma16_s((const void *)scalar_ptr(a.absum + (size_t)tok0 * nb_all * 16 + sbg * 16), (unsigned)(bt < last ? bt : last) * (unsigned)nb_all * 32u + (unsigned)(l & 1) * 16u,
                              dst + P2_BS + (unsigned)(4 * tw + wave) * 1024u);
            // (scales of 64 tokens: the upper half are the next wave's, with the same values)
            dma4_s((const void *)scalar_ptr(a.ad + (size_t)tok0 * nb_all + sbg), (unsigned)(yt < last ? yt : last) * (unsigned)nb_all * 4u, lds0 + P2_YD + (unsigned)((2 * y3 + tw) * P2_YDB + wave * 128));
        }
    };
    auto convert = [&](int buf) {                               // the wave's own share of the block sums, int16 -> f16 in place
        if (!MINS) return;
        uint8_t *q = smem_wg + buf * P2_BUF + P2_BS + (4 * tw + wave) * 1024 + lane * 16;
        const i16x8 v = *reinterpret_cast<const i16x8 *>(q);
        f16x8 f;
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = (_Float16)v[e];
        *reinterpret_cast<f16x8 *>(q) = f;
    };
    const unsigned b_off = (unsigned)lane * 16u;
    i32x4 B[8][2];                                              // [K-step][plane]
    u32x4 raw[4];                                               // codes, nibbles: as they are, of K-steps 2 c and 2 c + 1
    dma(0, 0, 0);
    typedef const __attribute__((address_space(1))) i32x4 g_i32x4;
    auto ld_b = [&](gbytes *blk, int j) {
        if (FORM != PF_CODES) {
            gbytes *q = blk + (FORM == PF_NIBBLES ? j : 2 * j) * 1024;
            asm("" : "+s"(q));
            if (!PACKED) B[j][0] = *(g_i32x4 *)(q + b_off);
            B[j][1] = *(g_i32x4 *)(q + b_off + (PACKED ? 0 : 1024));
        }
        if (PACKED && (j & 1)) {
            gbytes *q = blk + (FORM == PF_CODES ? j >> 1 : 8 + (j >> 1)) * 1024;
            asm("" : "+s"(q));
            raw[j >> 1] = __builtin_bit_cast(u32x4, *(g_i32x4 *)(q + b_off));
        }
    };
#pragma unroll
    for (int j = 0; j < 8; j++) { ld_b(blk0, j); __builtin_amdgcn_sched_barrier(0); }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    convert(0);
    __syncthreads();
    const bool nib = FORM == PF_MINS && __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int *>(smem_wg + P2_META + (SHARED ? 0 : tw * 2048) + 12));       // Q2_K planes: sixteen 4-bit mins

    i32x16 H[2], L[2];                                          // [tile parity]
    f32x16 ms;
    f32x4 yd = {0.0f, 0.0f, 0.0f, 0.0f};
    f16x8 as = {0, 0, 0, 0, 0, 0, 0, 0}, bm = as;
    float dd = 0.0f, ndm = 0.0f;
    // outputs 2 p, 2 p + 1 of a lane's sixteen of token tile t; ydn: where the tile's scales lie
    auto fold = [&](int t, int pr, int p, const uint8_t *ydp) {
#pragma unroll
        for (int r = 2 * p; r < 2 * p + 2; r++) {
            const float cf = (float)((H[pr][r] << SH) + L[pr][r]);
            if (MINS) facc[t][r] = fmaf(yd[r & 3], fmaf(dd, cf, ndm * ms[r]), facc[t][r]);
            else facc[t][r] = fmaf(yd[r & 3] * dd, cf, facc[t][r]);
        }
        if ((p & 1) && p < 7) yd = *reinterpret_cast<const f32x4 *>(ydp + (8 * ((p >> 1) + 1)) * 4);
    };
    // the block-sum term of the tile whose fold is next
    auto mins = [&]() {
        if (!MINS) return;
        f32x16 zf;
#pragma unroll
        for (int r = 0; r < 16; r++) zf[r] = 0.0f;
        ms = __builtin_amdgcn_mfma_f32_32x32x16_f16(as, bm, zf, 0, 0, 0);
    };
    int y3 = 0;                                                 // sb % 3: three sets of token scales, the last tile's fold reaches into the next super-block
    const uint8_t *yprev = sm_yd;
    for (int sb = 0; sb < nb; sb++) {
        const int sbuf = (sb & 1) * P2_BUF;
        const int nxt = sb + 1 < nb ? sb + 1 : sb, y3n = y3 == 2 ? 0 : y3 + 1;
        gbytes *blkn = blk0 + (size_t)nxt * BLOCK;
        const uint8_t *ys = sm_yd + y3 * 2 * P2_YDB + 16 * kg;
        unsigned x = (unsigned)(n * 256 + ((kg ^ (n & 15)) * 16));
        asm volatile("" : "+v"(x));
        auto ld_a = [&](int t, int j) { return *reinterpret_cast<const i32x4 *>(sm_a + sbuf + t * 8192 + (x ^ (unsigned)(32 * j))); };
        i32x4 A[2];
        u32x4 meta = *reinterpret_cast<const u32x4 *>(sm_meta + sbuf + (FORM == PF_CODES ? 512 : 0) + n * 16);
        A[0] = ld_a(0, 0); A[1] = ld_a(0, 1);
        uint32_t sw = 0;
        auto scales = [&](int c) { if (FORM == PF_CODES) sw = *reinterpret_cast<const uint32_t *>(sm_meta + sbuf + n * 16 + c * 4); };
        auto expand = [&](auto J) { constexpr int j = J.value; if constexpr (PACKED) expand_words<FORM, j>(raw[j >> 1], sw, B[j][0], B[j][1]); };
        scales(0);
        __builtin_amdgcn_sched_barrier(0);
        if (sb) {                                               // the last tile of the super-block before, while the operands come
            mins();
#pragma unroll
            for (int p = 0; p < 8; p++) fold(NT - 1, (NT - 1) & 1, p, yprev);
        }
        expand(std::integral_constant<int, 0>()); expand(std::integral_constant<int, 1>());
        scales(1);
        dd = h2f((uint16_t)(meta.x & 0xffff));
        asm("" : "+v"(dd));                                  // (as f32: folded into v_fma_mix_f32 it costs twice the issue slots)
        if (MINS) {
            ndm = -h2f((uint16_t)(meta.x >> 16));
            const unsigned w = kg ? meta.z : meta.y;            // mins 4 kg .. 4 kg + 3, each for two consecutive block sums
            if (nib) {                                          // eight 4-bit mins 8 kg .., one per block sum
#pragma unroll
                for (int e = 0; e < 8; e++) bm[e] = (_Float16)(float)((w >> (4 * e)) & 0xfu);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const _Float16 v = (_Float16)(float)((w >> (8 * e)) & 0xffu);
                    bm[2 * e] = v; bm[2 * e + 1] = v;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int pr = t & 1;
            if (t == (NT > 2 ? 1 : 0)) dma(nxt, (sb + 1) & 1, y3n);
            if (t == NT - 1) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile has landed; the planes' requests below stay in flight over the barrier
                convert((sb + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (t > 0 && j == 0) mins();
                if (j == 0) {
                    i32x16 z;
#pragma unroll
                    for (int r = 0; r < 16; r++) z[r] = 0;
                    H[pr] = mfma_i8(A[0], B[0][0], z); L[pr] = mfma_i8(A[0], B[0][1], z);
                } else { H[pr] = mfma_i8(A[j & 1], B[j][0], H[pr]); L[pr] = mfma_i8(A[j & 1], B[j][1], L[pr]); }
                if (j < 6) A[j & 1] = ld_a(t, j + 2);
                else if (t + 1 < NT) A[j & 1] = ld_a(t + 1, j - 6);
                if (MINS && j == 4) as = *reinterpret_cast<const f16x8 *>(sm_bs + sbuf + (32 * t + n) * 32 + kg * 16);
                if (PACKED && t == 0) {                         // two K-steps ahead
                    switch (j) {
                        case 0: expand(std::integral_constant<int, 2>()); break;
                        case 1: expand(std::integral_constant<int, 3>()); scales(2); break;
                        case 2: expand(std::integral_constant<int, 4>()); break;
                        case 3: expand(std::integral_constant<int, 5>()); scales(3); break;
                        case 4: expand(std::integral_constant<int, 6>()); break;
                        case 5: expand(std::integral_constant<int, 7>()); break;
                        default: break;
                    }
                }
                if (t == NT - 1) ld_b(blkn, j);
                if (t > 0) fold(t - 1, pr ^ 1, j, ys + (t - 1) * 128);
                if (j == 7) yd = *reinterpret_cast<const f32x4 *>(ys + t * 128);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        yprev = ys + (NT - 1) * 128;
        y3 = y3n;
        __syncthreads();
    }
    mins();
#pragma unroll
    for (int p = 0; p < 8; p++) fold(NT - 1, (NT - 1) & 1, p, yprev);
}

// SWIGLU: `planes` = ffn_gate, `planes_up` = ffn_up (n_rows rows each, same type): a workgroup takes 64 rows of BOTH (row-waves 0, 1 the
// gate rows, 2, 3 the same rows of up), the two waves of the same rows swap halves of their tiles through LDS at the end and store
// silu(gate . x) * (up . x) - one [T][n_rows] f32 result instead of two, and no separate SwiGLU pass over them.  ONE: one segment, known here (a struct made in the kernel and indexed
// at run time is scratch: 96 bytes a lane of mmq_planes2_moe_kernel)
template <int FORM, bool SWIGLU, bool ONE = SWIGLU>
__device__ __forceinline__ void planes2_body(const P2Args &a, const PlanesOut &po, int row_tile, int tok_tile, int n_tok_tiles, int zz) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb_all = a.K >> 8;
    const int sb_lo = (int)((long)nb_all * zz / a.n_split), nb = (int)((long)nb_all * (zz + 1) / a.n_split) - sb_lo;
    const int n_rows = a.n_rows, T = a.T;
    const int n_rt32 = (n_rows + 31) >> 5;
    const int rw = wave & 3, tw = wave >> 2;
    const int rt32 = SWIGLU ? row_tile * 2 + (rw & 1) : row_tile * 4 + rw;
    const uint8_t *base = SWIGLU && rw >= 2 ? a.planes_up : a.planes;
    const bool tile_ok = rt32 < n_rt32;
    // the batch's 32-token tiles, dealt evenly: to the workgroups' token tiles, and there to the two halves
    const int units = (T + 31) >> 5, per = (units + n_tok_tiles - 1) / n_tok_tiles, mine_u = units - tok_tile * per < per ? units - tok_tile * per : per;
    const int nt = mine_u <= 0 ? 0 : tw ? mine_u >> 1 : (mine_u + 1) >> 1;
    const int row0 = rt32 * 32, tok0 = (tok_tile * per + (tw ? (mine_u + 1) >> 1 : 0)) * 32, n = lane & 31, kg = lane >> 5, row = row0 + n;
    gbytes *blk0 = scalar_ptr(base + ((size_t)(tile_ok ? rt32 : n_rt32 - 1) * nb_all + sb_lo) * plane_block(FORM));
    float facc[4][16];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) facc[t][r] = 0.0f;
    // In mmq_planes2_kernel a half of fewer than four tiles fetches its rows' words itself (a second half of four means a first one): there the branch costs more than the requests, in gate | up and
    // the experts' launches, which fill the chip, less (us, once | by each half: 4096 x 14336 of Q6_K at 129 and 160 tokens 51.6 | 50.0, 53.5 | 51.1, of Q5_K at 80 37.8 | 36.5; gate | up of
    // 14336 x 4096 at 80 tokens of Q6_K 57.2 | 58.6, at 300 of Q5_K 107.9 | 109.6, at 1000 297 | 300).
#define P2_LOOP(NTV, FULLV) planes2_loop<FORM, NTV, FULLV, ONE || NTV == 4 || FORM == PF_CODES>(blk0, a, sb_lo, nb, tok0, tid, tw, smem, facc)
    if (nt == 4 && T - tok0 >= 128) P2_LOOP(4, true);
    else if (nt == 4) P2_LOOP(4, false);
    else if (nt == 3) P2_LOOP(3, false);
    else if (nt == 2) P2_LOOP(2, false);
    else if (nt == 1) P2_LOOP(1, false);
    else for (int i = 0; i <= nb; i++) __syncthreads();         // (a half without tokens keeps the barriers)
#undef P2_LOOP
    const bool all = nt == 4 && T - tok0 >= 128 && row0 + 32 <= n_rows;
    const int t_end = tok0 + 32 * nt < T ? tok0 + 32 * nt : T;  // tokens of this half: [tok0, t_end)
    auto token = [&](int t, int r) { return tok0 + 32 * t + (r & 3) + 8 * (r >> 2) + 4 * kg; };
    if (SWIGLU) {                                               // waves w (gate rows) and w + 2 (the same rows of up) swap halves: w finishes tokens 0 .. 63, w + 2 the others
        float *mine = reinterpret_cast<float *>(smem) + wave * 2048 + lane, *theirs = reinterpret_cast<float *>(smem) + (wave ^ 2) * 2048 + lane;
        auto give = [&](int t0) {
#pragma unroll
            for (int i = 0; i < 32; i++) mine[i * 64] = facc[t0 + (i >> 4)][i & 15];
        };
        auto finish = [&](int t0, bool all_) {
            float *out = po.out[0];
            const int ld_out = po.ld[0];
#pragma unroll
            for (int i = 0; i < 32; i++) {
                const int t = t0 + (i >> 4), gt = token(t, i & 15);
                const float own = facc[t][i & 15], oth = theirs[i * 64], gv = t0 ? oth : own, uv = t0 ? own : oth;
                const float y = (gv / (1.0f + expf(-gv))) * uv;
                if (all_ || (gt < t_end && row < n_rows)) out[(size_t)gt * ld_out + row] = y;
            }
        };
        if (rw < 2) give(2); else give(0);
        __syncthreads();
        if (!tile_ok) return;
        if (all) { if (rw < 2) finish(0, true); else finish(2, true); }
        else { if (rw < 2) finish(0, false); else finish(2, false); }
        return;
    }
    if (!tile_ok) return;
    int sg = 0;
    if (!ONE && po.n_seg > 1 && row0 >= po.row_end[0]) sg = 1;
    if (!ONE && po.n_seg > 2 && row0 >= po.row_end[1]) sg = 2;
    const bool split = a.n_split > 1;                           // partial sums of this K range: ws[zz][token][row], no residual
    float *out = split ? a.ws + (size_t)zz * T * n_rows : po.out[sg] - (sg ? po.row_end[sg - 1] : 0);
    const int ld_out = split ? n_rows : po.ld[sg];
    if (a.resid && !split) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float rv[16];                                       // (all requested before the first add)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int gt = token(t, r);
                rv[r] = a.resid[(size_t)(gt < T ? gt : T - 1) * ld_out + (row < n_rows ? row : n_rows - 1)];
            }
#pragma unroll
            for (int r = 0; r < 16; r++) facc[t][r] = rv[r] + facc[t][r];
        }
    }
    auto store = [&](bool all_) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int gt = token(t, r);
                if (all_ || (gt < t_end && row < n_rows)) out[(size_t)gt * ld_out + row] = facc[t][r];
            }
    };
    if (all) store(true); else store(false);
}

// MODE a PlaneForm, or P2_MIXED: per segment (po.form, of Q4_K, Q5_K or Q6_K; segment boundaries at multiples of 128 rows, so a workgroup's row tile is of one kind) - Q | K | V of
// the layers whose attn_v has more bits, in one launch.  The bodies lie behind workgroup-uniform branches (a run-time flag inside ONE body costs 92 bytes of scratch per lane and 2.3x the time).
constexpr int P2_MIXED = 4;
template <int MODE>
__global__ __launch_bounds__(NTHREADS) void mmq_planes2_kernel(const uint8_t *planes, int n_rows, int K, int T, int n_row_tiles, int n_tok_tiles,
                                                               const int8_t *aq, const float *ad, const int16_t *absum,
                                                               const PlanesOut po, const float *resid, float *ws, int n_split) {
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int tok_tile = loc % n_tok_tiles;
    const int zz = (loc / n_tok_tiles) % n_split;              // K split: partial sums go to ws[zz], mmq_splitk_reduce_kernel adds them up
    const int row_tile = (loc / (n_tok_tiles * n_split)) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;                       // workgroup-uniform
    P2Args a{planes, nullptr, n_rows, K, T, aq, ad, absum, resid, ws, n_split};
    if constexpr (MODE != P2_MIXED) planes2_body<MODE, false>(a, po, row_tile, tok_tile, n_tok_tiles, zz);
    else {
        int sg = 0;
        if (po.n_seg > 1 && row_tile * P2_ROWS >= po.row_end[0]) sg = 1;
        if (po.n_seg > 2 && row_tile * P2_ROWS >= po.row_end[1]) sg = 2;
        // where block 0 of the launch would lie if all were of this segment's form
        const int form = __builtin_amdgcn_readfirstlane(po.form[sg]);
        a.planes = planes + po.at[sg] - (size_t)(sg ? po.row_end[sg - 1] >> 5 : 0) * (size_t)(K >> 8) * plane_block(form);
        if (form == PF_SIGNED) planes2_body<PF_SIGNED, false>(a, po, row_tile, tok_tile, n_tok_tiles, zz);
        if (form == PF_CODES) planes2_body<PF_CODES, false>(a, po, row_tile, tok_tile, n_tok_tiles, zz);
        if (form == PF_NIBBLES) planes2_body<PF_NIBBLES, false>(a, po, row_tile, tok_tile, n_tok_tiles, zz);
    }
}

// ffn_gate and ffn_up with SwiGLU in the epilogue: n_rows rows of each, 64 per workgroup, out[t][row] = silu(gate) * up
template <int FORM>
__global__ __launch_bounds__(NTHREADS) void mmq_planes2_swiglu_kernel(const uint8_t *planes_gate, const uint8_t *planes_up, int n_rows, int K, int T,
                                                                      int n_row_tiles, int n_tok_tiles, const int8_t *aq, const float *ad,
                                                                      const int16_t *absum, const PlanesOut po) {
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int tok_tile = loc % n_tok_tiles;
    const int row_tile = (loc / n_tok_tiles) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;                       // workgroup-uniform
    planes2_body<FORM, true>(P2Args{planes_gate, planes_up, n_rows, K, T, aq, ad, absum, nullptr, nullptr, 1}, po, row_tile, tok_tile, n_tok_tiles, 0);
}

// ---- ggml_mul_mat_id on a prompt batch as ONE launch per projection.  The (token, rank) pairs of the batch are sorted by expert (moe_group_kernel: expert
// e owns rows [meta[NE + e], + meta[e]) of the grouped activation / result arrays); a workgroup is (row tile, token-tile slot j): slot j is the j-th 256-token tile
// of the concatenation of the experts' batches, found by walking the per-expert counts ON THE DEVICE - no host synchronisation to size per-expert launches, and
// eight half-empty launches of ~128 tokens become one that fills the chip.  The body is planes2_body: the wrapper hands it the expert's planes, the
// batch's rows as "the" token range (pointers offset to the batch's first row, T = the batch's length) and the tile index within the batch.
struct MoeTiles { const int32_t *meta; int n_expert; size_t plane_stride; };     // meta: [0, NE) tokens per expert, [NE, 2 NE) first grouped row
__device__ __forceinline__ bool moe_tile_of(const MoeTiles &m, int j, int &e_out, int &tile_out, int &r0_out, int &n_out) {
    for (int e = 0; e < m.n_expert; e++) {                      // (scalar: the counts are a few words of one cache line)
        const int n_e = __builtin_amdgcn_readfirstlane(m.meta[e]);
        const int tiles = (n_e + P2_TOK - 1) / P2_TOK;
        if (j < tiles) { e_out = e; tile_out = j; r0_out = __builtin_amdgcn_readfirstlane(m.meta[m.n_expert + e]); n_out = n_e; return true; }
        j -= tiles;
    }
    return false;
}
// an expert's rows of the grouped output
__device__ __forceinline__ PlanesOut moe_out(float *out, int ld_out, int r0, int n_rows) {
    PlanesOut po{};
    po.n_seg = 1; po.out[0] = out + (size_t)r0 * ld_out; po.ld[0] = ld_out; po.row_end[0] = n_rows;
    return po;
}
template <int FORM>
__global__ __launch_bounds__(NTHREADS) void mmq_planes2_swiglu_moe_kernel(const uint8_t *planes_gate, const uint8_t *planes_up, int n_rows, int K, int n_row_tiles,
                                                                          int n_tile_slots, const int8_t *aq, const float *ad, const int16_t *absum, float *out, int ld_out,
                                                                          const MoeTiles mt) {
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int slot = loc % n_tile_slots;
    const int row_tile = (loc / n_tile_slots) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;                       // workgroup-uniform
    int e, tile, r0, n_e;
    if (!moe_tile_of(mt, slot, e, tile, r0, n_e)) return;
    const size_t nb = (size_t)(K >> 8);
    const PlanesOut po = moe_out(out, ld_out, r0, n_rows);
    planes2_body<FORM, true>(P2Args{planes_gate + (size_t)e * mt.plane_stride, planes_up + (size_t)e * mt.plane_stride, n_rows, K, n_e,
                                    aq + (size_t)r0 * K, ad + (size_t)r0 * nb, absum + (size_t)r0 * (K >> 4), nullptr, nullptr, 1}, po, row_tile, tile, (n_e + P2_TOK - 1) / P2_TOK, 0);
}
template <int FORM>
__global__ __launch_bounds__(NTHREADS) void mmq_planes2_moe_kernel(const uint8_t *planes, int n_rows, int K, int n_row_tiles, int n_tile_slots,
                                                                   const int8_t *aq, const float *ad, const int16_t *absum, float *out, int ld_out, const MoeTiles mt) {
    const int bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3;
    const int slot = loc % n_tile_slots;
    const int row_tile = (loc / n_tile_slots) * 8 + xcd;
    if (row_tile >= n_row_tiles) return;
    int e, tile, r0, n_e;
    if (!moe_tile_of(mt, slot, e, tile, r0, n_e)) return;
    const size_t nb = (size_t)(K >> 8);
    const PlanesOut po = moe_out(out, ld_out, r0, n_rows);
    planes2_body<FORM, false, true>(P2Args{planes + (size_t)e * mt.plane_stride, nullptr, n_rows, K, n_e,
                                     aq + (size_t)r0 * K, ad + (size_t)r0 * nb, absum + (size_t)r0 * (K >> 4), nullptr, nullptr, 1}, po, row_tile, tile, (n_e + P2_TOK - 1) / P2_TOK, 0);
}

// out[t][row] = (resid) + ((part 0 + part 1) + (part 2 + part 3)) of ws[part][t][row] (a fixed order, so results do not depend on timing)
__global__ __launch_bounds__(256) void mmq_splitk_reduce_kernel(const float *ws, int n_split, int T, int n_rows, const PlanesOut po, const float *resid) {
    const size_t i4 = (size_t)blockIdx.x * 256 + threadIdx.x, per_tok = (size_t)n_rows >> 2;      // n_rows % 4 == 0 (launcher)
    if (i4 >= per_tok * T) return;
    const int t = (int)(i4 / per_tok), row = (int)(i4 % per_tok) * 4;
    const size_t plane = (size_t)T * n_rows, at = (size_t)t * n_rows + row;
    f32x4 v[4];                                                // (at most four parts; all requested before the first add)
#pragma unroll
    for (int z = 0; z < 4; z++) v[z] = *reinterpret_cast<const f32x4 *>(ws + (size_t)(z < n_split ? z : 0) * plane + at);
    f32x4 acc = v[0];
    if (n_split > 3) v[2] = v[2] + v[3];
    if (n_split > 1) acc = acc + v[1];
    if (n_split > 2) acc = acc + v[2];
    int sg = 0;
    if (po.n_seg > 1 && row >= po.row_end[0]) sg = 1;
    if (po.n_seg > 2 && row >= po.row_end[1]) sg = 2;
    float *o = po.out[sg] + (size_t)t * po.ld[sg] + (row - (sg ? po.row_end[sg - 1] : 0));
    if (resid) {
        const float *rp = resid + (size_t)t * po.ld[0] + row;
        acc.x = rp[0] + acc.x; acc.y = rp[1] + acc.y; acc.z = rp[2] + acc.z; acc.w = rp[3] + acc.w;
    }
    o[0] = acc.x; o[1] = acc.y; o[2] = acc.z; o[3] = acc.w;
}

// per-16 block sums of Q8_K split into int8 planes: bsum = 64*hi + lo, hi in [-32, 31], lo in [0, 63]
__global__ void mmq_prep_kernel(const int16_t *bsums, size_t n, int8_t *bh, int8_t *bl) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;     // over T * K/16
    if (i >= n) return;
    const int s = (int)bsums[i];
    const int hi = s >> 6;                    // arithmetic shift: floor(s / 64)
    bh[i] = (int8_t)hi;
    bl[i] = (int8_t)(s - 64 * hi);
}

template <int TYPE, int MT>
hipError_t launch_one(const uint8_t *W, size_t row_bytes, int n_rows, int K, int T, const ActQuant &q, const int8_t *bh, const int8_t *bl,
                      float *out, int ld_out, const float *resid, hipStream_t st) {
    using G = Geo<MT>;
    const int nrt = (n_rows + G::ROW_TILE - 1) / G::ROW_TILE, ntt = (T + G::TOK_TILE - 1) / G::TOK_TILE;
    const int groups = (nrt + 7) / 8;                                   // row tiles in groups of 8 (one per XCD)
    const dim3 grid((unsigned)(groups * ntt * 8));
    hipLaunchKernelGGL((mmq_kernel<TYPE, MT>), grid, dim3(NTHREADS), (size_t)G::LDS_BYTES, st, W, row_bytes, n_rows, K, T, nrt, ntt,
                       q.qs, q.d, bh, bl, out, ld_out, resid);
    return hipGetLastError();
}

int g_mmq_mt = 0;   // 0 = by T; tools may force 1 / 2 / 4
int g_mmq_split = 0;   // tools: force the K split of the 128 x 256 kernel (0 = by shape, 1 = none)
int g_mmq_p2 = -1;     // tools: 0 = never the 128 x 256 kernel, 1 = by shape, -1 = MI355_MMQ_PLANES2 / default

template <int TYPE>
hipError_t launch_type(const uint8_t *W, size_t row_bytes, int n_rows, int K, int T, const ActQuant &q, const int8_t *bh, const int8_t *bl,
                       float *out, int ld_out, const float *resid, hipStream_t st) {
    // one token tile per wave: the expansion is VALU-bound and larger tiles spill (measured 34 ms vs 40 ms per 512-token
    // prompt of the 8B model); MI355_MMQ_MT / mmq_set_tiles(2) select the 128 x 128 workgroup tile
    static const int env_mt = getenv("MI355_MMQ_MT") ? atoi(getenv("MI355_MMQ_MT")) : 0;
    int mt = 1;
    if (env_mt == 1 || env_mt == 2) mt = env_mt;
    if (g_mmq_mt == 1 || g_mmq_mt == 2) mt = g_mmq_mt;
    switch (mt) {
        case 2: return launch_one<TYPE, 2>(W, row_bytes, n_rows, K, T, q, bh, bl, out, ld_out, resid, st);
        default: return launch_one<TYPE, 1>(W, row_bytes, n_rows, K, T, q, bh, bl, out, ld_out, resid, st);
    }
}

}  // namespace

void mmq_set_tiles(int mt) { g_mmq_mt = mt; }
void mmq_set_split(int n) { g_mmq_split = n; }
void mmq_set_lds_form(int on) { g_mmq_p2 = on; }

// continuous-batching decode steps and prompts up to a few hundred tokens: 3 <= T <= g_ksplit_max.  This kernel reads the GGUF bytes (0.56 B / weight) and expands them in
// registers, once per 64 tokens; the planes kernels read 0.6 to 2 B / weight that they need expand less or not at all, the fewer times the more tokens there are.  Behind 256 tokens every tensor with
// planes goes to them: a whole 8B prompt of 320 tokens took 17.2 ms here and 15.2 there, of 384 19.1 and 15.5, before the tiles became faster.
static int g_ksplit_max = getenv("MI355_KSPLIT_MAX") ? atoi(getenv("MI355_KSPLIT_MAX")) : 256;
bool mmq_ksplit_applicable(int type, int K, int T) {
    // from 3 tokens: the mat-vec takes 4 + 2 + 1 tokens per pass over the weights, so 3 sequences cost 4.5 ms and 6 cost 6.4 ms a step against
    // 3.7 ms through this kernel.  Two go to mmq_few.hip or stay with the mat-vec (mmq_few_pair)
    return (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && (K % 256) == 0 && T >= 3 && T <= g_ksplit_max;
}

static int planes2_split(int n_rows, int K, int T, const MMQWorkspace &wsp, bool *takes);
// Which kernel takes a launch of 65 .. 256 tokens is a matter of shape (to 64 tokens mmq_few_takes chooses): this one, or the 128 x 256 tiles, K split over the workgroups where the
// workspace allows it.  The choice is by the two launches' times.  Both are whole rounds of one workgroup a CU, and a round is its super-blocks and a start (us): K-split, 32 rows x 64
// tokens, an eighth of the super-blocks of 5.2 and 3.5; tiles, the part's super-blocks of 1.5 + T / 128, to 128 tokens of Q6_K, which they read as two bytes a weight, 2 + T / 128, and 7, and 4
// more where the parts' sum is a launch of its own.
// From 97 to 128 tokens a workgroup has four tiles of 32 and takes as long as at 128: gate | up of 5632 x 2048, Q4_K, at 100 tokens 24.4 / 27.0, ten layers of it at 97, 100 and 112 with the
// tiles 929, 933, 940 us and without 905, 911, 919.
// Measured with weights from HBM, Q4_K, K-split / tiles without the sum's launch, at 72, 128 and 256 tokens (Q5_K costs either kernel a tenth more):
//   2048 x 2048   9/13 9/15 10/18     2048 x 5632  18/18 19/20 20/24    1536 x 8960   23/23 27/27 26/34     gate | up of 5632 x 2048    25/24 25/27 44/32
//   3072 x 3072  11/14 12/16 19/19    3072 x 8192  24/22 24/25 43/31    5120 x 5120   28/17 28/19 42/24     gate | up of 8192 x 3072    40/32 41/37 74/44
//   4096 x 4096  15/15 15/16 26/20    6144 x 4096  25/15 25/17 37/21    4096 x 14336  40/35 40/40 72/50     gate | up of 14336 x 4096   89/43 91/49 166/61
// Q6_K at 65, 96 and 128 tokens:  2048 x 5632  20/21 20/21 20/23    4096 x 14336  46/45 43/45 43/47    3584 x 18944  55/55 53/57 54/59    6144 x 4096  27/19 27/20 27/21
//   gate | up of 5632 x 2048  25/28 25/28 25/30    of 8192 x 3072  43/41 43/41 44/43    of 14336 x 4096  101/58 95/56 96/61
// (tiles of planes, before Q4_K came as codes: gate | up of 14336 x 4096 at 130 tokens 70, 6144 x 4096 25.)  Whole prompts of eight layers of an 8B model, us, K-split to 128 tokens and now:
// 65 tokens 1624, 1083; 96 1672, 1128; 128 1727, 1227.
static bool tiles_beat_ksplit(int type, int n_rows, int K, int T, MMQWorkspace wsp, bool pair, bool sum_free) {
    bool takes = false;
    const int rows = pair ? 2 * n_rows : n_rows, parts = planes2_split(rows, K, T, pair ? MMQWorkspace() : wsp, &takes), nb = K >> 8;
    if (!takes) return n_rows >= 8192 && !(pair && T <= 128);  // (then the planes kernel below, by rows; ffn_gate | ffn_up are one launch here and two there)
    const auto up = [](long a, long b) { return (double)((a + b - 1) / b); };
    const double here = up(up(rows, 32) * up(T, 64), num_cu()) * (5.2 * nb / 8 + 3.5);
    const double tiles = up(up(rows, P2_ROWS) * up(T, P2_TOK) * parts, num_cu()) * (((type == T_Q6_K && T <= 128 ? 2.0 : 1.5) + (T > 96 && T < 128 ? 128 : T) / 128.0) * up(nb, parts) + 7.0) + (parts > 1 && !sum_free ? 4.0 : 0.0);
    return tiles < here;
}
bool mmq_ksplit_preferred(int type, int n_rows, int K, int T, bool has_planes, MMQWorkspace wsp, bool sum_free, bool pair) {
    static const int env = getenv("MI355_KSPLIT_SHAPE") ? atoi(getenv("MI355_KSPLIT_SHAPE")) : 1;
    if (!mmq_ksplit_applicable(type, K, T)) return false;
    if (!env || !has_planes || !mmq_applicable(type, K, T)) return true;
    return T <= 64 || !tiles_beat_ksplit(type, n_rows, K, T, wsp, pair, sum_free);
}

// segs: up to 3 tensors sharing the activation; swiglu (to 32 tokens, or where mmq_few_takes): segs = {gate, up} of one type and shape, out = silu(gate.x) * (up.x) into segs[0].out
hipError_t launch_mmq_ksplit_multi(const MMQSeg *segs, int n_seg, int K, int T, const ActQuant &q, const int8_t *bh, const int8_t *bl,
                                   bool swiglu, hipStream_t st) {
    if (n_seg < 1 || n_seg > 3) return hipErrorInvalidValue;
    if (swiglu && (n_seg != 2 || segs[0].type != segs[1].type || segs[0].n_rows != segs[1].n_rows)) return hipErrorInvalidValue;
    if (mmq_few_takes(segs, n_seg, K, T, q, swiglu)) return launch_mmq_few(segs, n_seg, K, T, q, swiglu, st);
    KSplitArgs a{};
    a.n_seg = n_seg; a.K = K; a.T = T; a.swiglu = swiglu ? 1 : 0;
    a.aq = q.qs; a.ad = q.d; a.abh = bh; a.abl = bl;
    int tiles = 0;
    for (int i = 0; i < n_seg; i++) {
        a.seg[i] = segs[i];
        a.seg[i].tile0 = tiles;
        if (!swiglu || i == 0) tiles += (segs[i].n_rows + 31) / 32;
    }
    const int mt = T <= 32 ? 1 : 2;
    if (swiglu && mt > 1) return hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles, (unsigned)((T + 32 * mt - 1) / (32 * mt)));
#define KS(MTV, SW)                                                                                                  \
    {                                                                                                                \
        constexpr int TOKV = 32 * MTV;                                                                               \
        size_t lds = (size_t)8 * (TOKV * A_STRIDE + 2 * TOKV * 16 + TOKV * 4);                                        \
        const size_t red = (size_t)8 * (SW ? 2 : 1) * MTV * 16 * 64 * 4;                                             \
        if (red > lds) lds = red;                                                                                    \
        if (lds > 65536) (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_ksplit_kernel<MTV, SW>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        hipLaunchKernelGGL((mmq_ksplit_kernel<MTV, SW>), grid, dim3(NTHREADS), lds, st, a);                          \
    }
    if (swiglu) KS(1, true)
    else if (mt == 1) KS(1, false) else KS(2, false)
#undef KS
    return hipGetLastError();
}

size_t mmq_planes_bytes(int type, int64_t n_rows, int K) {
    if ((type != T_Q4_K && type != T_Q5_K && type != T_Q6_K && type != T_Q2_K && type != T_Q3_K) || (K % 256) != 0) return 0;
    return (size_t)((n_rows + 31) / 32) * (size_t)(K >> 8) * plane_block(plane_form(type));
}

bool mmq_planes_same_form(int type_a, int type_b) { return plane_form(type_a) == plane_form(type_b); }

hipError_t launch_mmq_expand(int type, const uint8_t *W, size_t row_bytes, int n_rows, int K, uint8_t *planes, hipStream_t st) {
    const int nb = K >> 8, n_rt = (n_rows + 31) / 32;
    const dim3 grid((unsigned)((n_rt * nb + 3) / 4));
    switch (type) {
        case T_Q4_K: hipLaunchKernelGGL(mmq_pack_kernel<T_Q4_K>, grid, dim3(256), 0, st, W, row_bytes, n_rows, nb, n_rt, planes); break;
        case T_Q5_K: hipLaunchKernelGGL(mmq_pack_kernel<T_Q5_K>, grid, dim3(256), 0, st, W, row_bytes, n_rows, nb, n_rt, planes); break;
        case T_Q6_K: hipLaunchKernelGGL(mmq_expand_kernel, grid, dim3(256), 0, st, W, row_bytes, n_rows, nb, n_rt, planes); break;
        case T_Q2_K: hipLaunchKernelGGL(mmq_expand_small_kernel<T_Q2_K>, grid, dim3(256), 0, st, W, row_bytes, n_rows, nb, n_rt, planes); break;
        case T_Q3_K: hipLaunchKernelGGL(mmq_expand_small_kernel<T_Q3_K>, grid, dim3(256), 0, st, W, row_bytes, n_rows, nb, n_rt, planes); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_mmq_planes(int type, const uint8_t *planes, int n_rows, int K, int T, const ActQuant &q, const int8_t *bh, const int8_t *bl,
                             float *out, int ld_out, const float *resid, hipStream_t st, MMQWorkspace wsp, int *parts) {
    return launch_mmq_planes_multi(type, planes, &n_rows, &out, &ld_out, 1, K, T, q, bh, bl, resid, st, wsp, nullptr, parts);
}

// the K split the 128 x 256 kernel would run a tensor (or concatenation) of n_rows rows with, and whether it takes the launch at all
static int planes2_split(int n_rows, int K, int T, const MMQWorkspace &wsp, bool *takes) {
    static const int env_mt = getenv("MI355_MMQ_MT") ? atoi(getenv("MI355_MMQ_MT")) : 0;
    static const int env_p2_0 = getenv("MI355_MMQ_PLANES2") ? atoi(getenv("MI355_MMQ_PLANES2")) : 1;
    const int env_p2 = g_mmq_p2 >= 0 ? g_mmq_p2 : env_p2_0;
    static const int env_sk = getenv("MI355_MMQ_SPLITK") ? atoi(getenv("MI355_MMQ_SPLITK")) : -1;   // 0 off, 2..4 forced
    const int nb = K >> 8;
    const long wg = (long)((n_rows + P2_ROWS - 1) / P2_ROWS) * ((T + P2_TOK - 1) / P2_TOK);
    // One workgroup fills a CU, so K is split while the parts still run side by side - at least four super-blocks each, for a workgroup's start and end cost two.  us a launch
    // (Q4_K; unsplit / by this rule / one part more; the planes kernel below): 4096 x 4096 at 160, 512, 611, 1280 tokens 55 / 27 / -, 62 / 38 / -, 61 / 46 / 64,
    // 71 / 71 / 92 against 53, 48, 78, 126; 4096 x 14336: 169 / 59 / -, 205 / 82 / -, 189 / 114 / 158, 217 / 217 / 247 against 145, 144, 249, 396;
    // 6144 x 4096 at 160 and 512: 57 / 33 / -, 66 / 50 / 71 against 50, 93; 22016 x 4096 at 160 and 512: 63 / 63 / 81, 141 / 141 / 149 against 99, 213.
    int n_split = 1;
    if (g_mmq_split > 1 || env_sk > 1) n_split = g_mmq_split > 1 ? g_mmq_split : env_sk;
    else if (env_sk != 0 && g_mmq_split != 1) n_split = (int)std::max(1L, std::min({num_cu() / wg, 4L, (long)nb / 4}));
    n_split = std::min({n_split, nb, 4});                       // (the reductions add four parts at most)
    if (n_split < 1 || (n_rows % 4) != 0 || !wsp.p || (size_t)n_split * T * n_rows * sizeof(float) > wsp.bytes) n_split = 1;
    // (an unsplit launch wants a third of the CUs: 11264 x 2048 at 160 and 256 tokens - 88 workgroups - 35 and 40 us against 31 and 56, 4096 x 4096 at 300 - 64 - 53 against 47)
    *takes = g_mmq_mt == 4 || (g_mmq_mt == 0 && env_mt == 0 && env_p2 != 0 && T > 64 && (n_split > 1 || wg * 3 >= num_cu()));
    return n_split;
}

// Segments of several forms in one launch: only the 128 x 256 kernel has that form, and segments must end on its row tiles
bool mmq_planes_mixed_ok(const int *seg_rows, int n_seg, int K, int T, MMQWorkspace wsp) {
    static const bool env_on = !(getenv("MI355_MMQ_MIXED") && getenv("MI355_MMQ_MIXED")[0] == '0');
    if (!env_on) return false;
    int n_rows = 0;
    for (int i = 0; i < n_seg; i++) { if (i + 1 < n_seg && (seg_rows[i] % P2_ROWS) != 0) return false; n_rows += seg_rows[i]; }
    bool takes = false;
    (void)planes2_split(n_rows, K, T, wsp, &takes);
    return takes && n_seg >= 1 && n_seg <= 3;
}

// ffn_gate | ffn_up of one plane type with SwiGLU in the epilogue: 64 rows of each per workgroup
bool mmq_planes_swiglu_ok(int type_gate, int type_up, int n_rows, int K, int T) {
    static const bool env_on = !(getenv("MI355_MMQ_SWIGLU") && getenv("MI355_MMQ_SWIGLU")[0] == '0');
    if (!env_on || type_gate != type_up || mmq_planes_bytes(type_gate, n_rows, K) == 0 || (n_rows % 32) != 0) return false;
    bool takes = false;
    (void)planes2_split(2 * n_rows, K, T, MMQWorkspace(), &takes);
    return takes;
}

hipError_t launch_mmq_planes_swiglu(int type, const uint8_t *planes_gate, const uint8_t *planes_up, int n_rows, int K, int T, const ActQuant &q,
                                    float *out, int ld_out, hipStream_t st) {
    if (!mmq_planes_swiglu_ok(type, type, n_rows, K, T)) return hipErrorInvalidValue;
    PlanesOut po{};
    po.n_seg = 1; po.out[0] = out; po.ld[0] = ld_out; po.row_end[0] = n_rows;
    const int nrt = (n_rows + 63) / 64, ntt = (T + P2_TOK - 1) / P2_TOK;
    const dim3 grid((unsigned)(((nrt + 7) / 8) * ntt * 8));
#define GO(F) { (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_planes2_swiglu_kernel<F>), hipFuncAttributeMaxDynamicSharedMemorySize, P2_LDS); \
                hipLaunchKernelGGL((mmq_planes2_swiglu_kernel<F>), grid, dim3(NTHREADS), (size_t)P2_LDS, st, planes_gate, planes_up, n_rows, K, T, nrt, ntt, q.qs, q.d, q.bsums, po); }
    switch (plane_form(type)) {
        case PF_CODES: GO(PF_CODES) break;
        case PF_NIBBLES: GO(PF_NIBBLES) break;
        case PF_MINS: GO(PF_MINS) break;
        default: GO(PF_SIGNED) break;
    }
#undef GO
    return hipGetLastError();
}

// the grouped (all experts, one launch) forms: `rows_max` = rows of the grouped arrays (tokens x experts used), meta = moe_group_kernel's counts and offsets
bool mmq_planes_moe_ok(int type, int n_rows, int K) {
    static const bool env_on = !(getenv("MI355_MOE_GROUPED_LAUNCH") && getenv("MI355_MOE_GROUPED_LAUNCH")[0] == '0');
    return env_on && (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && mmq_planes_bytes(type, n_rows, K) != 0 && (n_rows % 128) == 0 && (K % 256) == 0;
}
hipError_t launch_mmq_planes_swiglu_moe(int type, const uint8_t *planes_gate, const uint8_t *planes_up, size_t plane_stride, int n_expert, const int32_t *meta,
                                        int n_rows, int K, int rows_max, const ActQuant &q, float *out, int ld_out, hipStream_t st) {
    if (!mmq_planes_moe_ok(type, n_rows, K) || n_expert < 1 || !meta || !q.qs || !q.d || !q.bsums) return hipErrorInvalidValue;
    const int nrt = (n_rows + 63) / 64, slots = (rows_max + P2_TOK - 1) / P2_TOK + n_expert;     // every expert may end in a partial tile
    const dim3 grid((unsigned)(((nrt + 7) / 8) * slots * 8));
    const MoeTiles mt{meta, n_expert, plane_stride};
#define GO(F) { (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_planes2_swiglu_moe_kernel<F>), hipFuncAttributeMaxDynamicSharedMemorySize, P2_LDS); \
                hipLaunchKernelGGL((mmq_planes2_swiglu_moe_kernel<F>), grid, dim3(NTHREADS), (size_t)P2_LDS, st, planes_gate, planes_up, n_rows, K, nrt, slots, q.qs, q.d, q.bsums, out, ld_out, mt); }
    switch (plane_form(type)) {
        case PF_CODES: GO(PF_CODES) break;
        case PF_NIBBLES: GO(PF_NIBBLES) break;
        default: GO(PF_SIGNED) break;
    }
#undef GO
    return hipGetLastError();
}
hipError_t launch_mmq_planes_moe(int type, const uint8_t *planes, size_t plane_stride, int n_expert, const int32_t *meta, int n_rows, int K, int rows_max,
                                 const ActQuant &q, float *out, int ld_out, hipStream_t st) {
    if (!mmq_planes_moe_ok(type, n_rows, K) || n_expert < 1 || !meta || !q.qs || !q.d || !q.bsums) return hipErrorInvalidValue;
    const int nrt = (n_rows + P2_ROWS - 1) / P2_ROWS, slots = (rows_max + P2_TOK - 1) / P2_TOK + n_expert;
    const dim3 grid((unsigned)(((nrt + 7) / 8) * slots * 8));
    const MoeTiles mt{meta, n_expert, plane_stride};
#define GO(F) { (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_planes2_moe_kernel<F>), hipFuncAttributeMaxDynamicSharedMemorySize, P2_LDS); \
                hipLaunchKernelGGL((mmq_planes2_moe_kernel<F>), grid, dim3(NTHREADS), (size_t)P2_LDS, st, planes, n_rows, K, nrt, slots, q.qs, q.d, q.bsums, out, ld_out, mt); }
    switch (plane_form(type)) {
        case PF_CODES: GO(PF_CODES) break;
        case PF_NIBBLES: GO(PF_NIBBLES) break;
        default: GO(PF_SIGNED) break;
    }
#undef GO
    return hipGetLastError();
}

hipError_t launch_mmq_planes_multi(int type, const uint8_t *planes, const int *seg_rows, float *const *outs, const int *lds_out, int n_seg, int K, int T,
                                   const ActQuant &q, const int8_t *bh, const int8_t *bl, const float *resid, hipStream_t st, MMQWorkspace wsp,
                                   const int *seg_types, int *parts) {
    if (n_seg < 1 || n_seg > 3 || (n_seg > 1 && resid)) return hipErrorInvalidValue;
    PlanesOut po{};
    po.n_seg = n_seg;
    int n_rows = 0;
    bool mixed = false, mins = false;
    size_t at = 0;
    for (int i = 0; i < n_seg; i++) {
        if (i + 1 < n_seg && (seg_rows[i] % 32) != 0) return hipErrorInvalidValue;
        n_rows += seg_rows[i];
        po.out[i] = outs[i]; po.ld[i] = lds_out[i]; po.row_end[i] = n_rows;
        const int ti = seg_types ? seg_types[i] : type;
        po.form[i] = plane_form(ti);
        po.at[i] = at;
        at += (mmq_planes_bytes(ti, seg_rows[i], K) + 255) & ~(size_t)255;
        mixed = mixed || po.form[i] != plane_form(type);
        mins = mins || po.form[i] == PF_MINS;
    }
    if (mixed && (mins || !mmq_planes_mixed_ok(seg_rows, n_seg, K, T, wsp))) return hipErrorInvalidValue;
    static const int env_mt = getenv("MI355_MMQ_MT") ? atoi(getenv("MI355_MMQ_MT")) : 0;
    // 128 x 128 workgroup tiles (two token tiles per wave) when that still yields ~2 workgroups per CU, else 256 x 32
    // tiles, which quadruple the workgroup count (measured on the 8B shapes: gate/up 297 vs 383 us, N = 4096 tensors
    // 54-144 vs 75-204 us per layer)
    const long wg2 = (long)((n_rows + 127) / 128) * ((T + 127) / 128);
    int mt = (T <= 32 || wg2 < 3L * num_cu() / 2) ? 1 : 2;
    if (n_seg > 1 && T > 32 && wg2 * 4 >= 3L * num_cu()) mt = 2;       // concatenated Q | K | V: 192 workgroups of 128 x 128 beat 384 of 256 x 32 (59 vs 71 us)
    if (env_mt == 1 || env_mt == 2) mt = env_mt;
    if (g_mmq_mt == 1 || g_mmq_mt == 2) mt = g_mmq_mt;
    // 128 rows x 256 tokens per workgroup from 65 tokens on; tensors with too few rows to cover the chip that way split K over 2..4 workgroups (partial sums in
    // the caller's workspace, added up pairwise)
    bool p2 = false;
    const int n_split = planes2_split(n_rows, K, T, wsp, &p2);
    if (p2) {
        const int nrt = (n_rows + P2_ROWS - 1) / P2_ROWS, ntt = (T + P2_TOK - 1) / P2_TOK;
        const dim3 grid((unsigned)(((nrt + 7) / 8) * ntt * n_split * 8));
#define GO(M) { (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_planes2_kernel<M>), hipFuncAttributeMaxDynamicSharedMemorySize, P2_LDS); \
                hipLaunchKernelGGL((mmq_planes2_kernel<M>), grid, dim3(NTHREADS), (size_t)P2_LDS, st, planes, n_rows, K, T, nrt, ntt, q.qs, q.d, q.bsums, po, resid, wsp.p, n_split); }
        if (mixed) GO(P2_MIXED)
        else switch (plane_form(type)) {
            case PF_CODES: GO(PF_CODES) break;
            case PF_NIBBLES: GO(PF_NIBBLES) break;
            case PF_MINS: GO(PF_MINS) break;
            default: GO(PF_SIGNED) break;
        }
#undef GO
        if (n_split > 1 && parts) *parts = n_split;
        else if (n_split > 1) {
            const size_t n4 = (size_t)T * (n_rows >> 2);
            hipLaunchKernelGGL(mmq_splitk_reduce_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, wsp.p, n_split, T, n_rows, po, resid);
        }
        return hipGetLastError();
    }
#define PLN(FORMV, MTV)                                                                                                   \
    {                                                                                                                     \
        using G = Geo<MTV>;                                                                                               \
        const int nrt = (n_rows + G::ROW_TILE - 1) / G::ROW_TILE, ntt = (T + G::TOK_TILE - 1) / G::TOK_TILE;              \
        const dim3 grid((unsigned)(((nrt + 7) / 8) * ntt * 8));                                                           \
        const size_t lds2 = 2 * (size_t)G::LDS_BYTES;                                                                     \
        if (lds2 > 65536) (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&mmq_planes_kernel<FORMV, MTV>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds2); \
        hipLaunchKernelGGL((mmq_planes_kernel<FORMV, MTV>), grid, dim3(NTHREADS), lds2, st, planes, n_rows, K, T, nrt, ntt, \
                           q.qs, q.d, bh, bl, po, resid);                                                                 \
    }
    switch (plane_form(type)) {
        case PF_CODES: if (mt == 1) PLN(PF_CODES, 1) else PLN(PF_CODES, 2) break;
        case PF_NIBBLES: if (mt == 1) PLN(PF_NIBBLES, 1) else PLN(PF_NIBBLES, 2) break;
        case PF_MINS: if (mt == 1) PLN(PF_MINS, 1) else PLN(PF_MINS, 2) break;
        default: if (mt == 1) PLN(PF_SIGNED, 1) else PLN(PF_SIGNED, 2) break;
    }
#undef PLN
    return hipGetLastError();
}

bool mmq_applicable(int type, int K, int T) {
    return (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && (K % 256) == 0 && T >= 32 && (size_t)T * (size_t)K < (1ull << 32);
}
size_t mmq_prep_bytes(int K, int T) { return (size_t)T * (K >> 4); }

hipError_t launch_mmq_prep(const ActQuant &q, int K, int T, int8_t *bh, int8_t *bl, hipStream_t st) {
    const size_t n = (size_t)T * (K >> 4);
    hipLaunchKernelGGL(mmq_prep_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, q.bsums, n, bh, bl);
    return hipGetLastError();
}

// out[t * ld_out + r] = (resid ? resid[...] : 0) + dot(W[r], act[t]);  bh/bl from launch_mmq_prep
hipError_t launch_mmq(int type, const uint8_t *W, size_t row_bytes, int n_rows, int K, int T, const ActQuant &q,
                      const int8_t *bh, const int8_t *bl, float *out, int ld_out, const float *resid, hipStream_t st) {
    switch (type) {
        case T_Q4_K: return launch_type<T_Q4_K>(W, row_bytes, n_rows, K, T, q, bh, bl, out, ld_out, resid, st);
        case T_Q5_K: return launch_type<T_Q5_K>(W, row_bytes, n_rows, K, T, q, bh, bl, out, ld_out, resid, st);
        case T_Q6_K: return launch_type<T_Q6_K>(W, row_bytes, n_rows, K, T, q, bh, bl, out, ld_out, resid, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mi355
