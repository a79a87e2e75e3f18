// mmq_few.hip — the K-split contraction of 3 .. 64 tokens  Y[t][r] = dot(W[r,:], act_q8K[t,:])  (continuous-batching ticks, the short turn of a conversation):
// K-quant weights in their GGUF form, Q8_K activations, int8 matrix cores, the integer of ggml_vec_dot_q{4,5,6}_K_q8_K per (row, token, super-block).
//
// What bounds it: the weights, read once from HBM (0.56 .. 0.82 B each), and in front of them the ~140 vector instructions per unit and token tile below (matrix
// pipe and memory idle half of the time at two waves per SIMD).  Measured on an 8B Q4_K_M model, kernel times before -> now: gate | up (66 MB) at 4 tokens
// 27.2 -> 18.7 us, at 37 tokens 51.4 -> 37.0; attn_output and ffn_down together 19.1 -> 12.3 a launch at 4; the head (431 MB) 129 -> 98; before is the 32 x 32
// form of mmq.hip, whose waves had no load in flight while they computed and which left half of the CUs without a row tile.
//   * A unit of work is 16 weight rows x one super-block (v_mfma_i32_16x16x32_i8: M = 16 tokens, N = 16 rows, K = the 32 weights of one scale group of Q4_K / Q5_K):
//     a 4096-row tensor is 256 row tiles, one per CU, and 16 tokens pad to 16, 37 to 48.
//   * One workgroup per CU walks its row tiles; its eight waves take a tile's super-blocks round-robin, and the weights of the next PD units - of the next tile
//     too - are in flight in registers while one is worked on.
//   * A wave asks for a unit as whole pieces of its rows, 144 (176, 208) consecutive bytes per row and super-block, and turns it into operands through LDS of its
//     own (a row's stride of 36, 44 or 52 words: no bank conflicts, no barrier).  Asked for as operands directly - 32 bytes of sixteen rows per request - every
//     128-byte line is asked for by four or five requests: gate | up of an 8B layer took 29 us that way.
//   * The activations come as operand blocks laid out by the quantiser (ActQuant::qf).  Read from rows of K bytes instead, sixteen lanes hit sixteen lines a power
//     of two apart: 34 us at 4 tokens, 43 at 16.  A wave meets the same super-blocks in every tile: up to 4096 columns and 32 tokens they stay in registers.
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
typedef short i16x2 __attribute__((ext_vector_type(2)));

constexpr int NW = 8, NT = 64 * NW;

__device__ __forceinline__ u32x4 ldg16(const void *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ u32x2 ldg8(const void *p) { return *reinterpret_cast<const u32x2 *>(p); }
__device__ __forceinline__ long as_long(u32x2 v) { return __builtin_bit_cast(long, v); }
__device__ __forceinline__ i32x4 mfma32(u32x2 a, u32x2 b, i32x4 c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(as_long(a), as_long(b), c, 0, 0, 0); }

// A unit, 16 rows x one super-block, as it is asked for: piece p = lane + 64 i is 16 bytes of row p / PIECES; rows past the end read the last one (never stored)
template <int TYPE> struct Raw {
    static constexpr int PIECES = TYPE == T_Q4_K ? 9 : TYPE == T_Q5_K ? 11 : 13, N = (16 * PIECES + 63) / 64, LDS = N * 1024, STRIDE = 16 * PIECES;
    u32x4 v[N];
    uint32_t d16 = 0;                                        // Q6_K: the row's scale, which lies apart
    __device__ __forceinline__ void load(const uint8_t *W, int rows, unsigned row_bytes, int nb, int sb, int lane) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int q = lane + 64 * i, p = q < STRIDE ? q : 0, r = p / PIECES, c = p - r * PIECES;    // (lanes past the unit: its first piece)
            unsigned o = (unsigned)(r < rows ? r : rows - 1) * row_bytes;
            if constexpr (TYPE == T_Q6_K)                    // row planes: ql (8 pieces), qh (4), scales (1)
                o += c < 8 ? (unsigned)sb * 128u + 16u * c : c < 12 ? (unsigned)nb * 128u + (unsigned)sb * 64u + 16u * (c - 8) : (unsigned)nb * 192u + (unsigned)sb * 16u;
            else o += (unsigned)sb * (unsigned)STRIDE + 16u * c;
            v[i] = ldg16(W + o);
        }
        if constexpr (TYPE == T_Q6_K) {
            const int r = lane & 15;
            d16 = *reinterpret_cast<const uint16_t *>(W + (unsigned)(r < rows ? r : rows - 1) * row_bytes + (unsigned)nb * 208u + (unsigned)sb * 2u);
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
    static constexpr bool GROUPS = true;
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
    static constexpr bool GROUPS = true;
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
    static constexpr bool GROUPS = false;                    // (two scales per step)
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
// pair (2 S, 2 S + 1) of scale groups per 16 bytes -, its block sums' two int8 planes, and the block scales of the four tokens whose results the lane holds
template <int MT> struct Act {
    u32x4 a[MT][4];
    u32x2 bh[MT], bl[MT];
    f32x4 yd[MT];
    __device__ __forceinline__ void load(const uint8_t *qf, int tile0, int nb, int sb, int lane, int n) {    // the first n of the tiles
#pragma unroll
        for (int t = 0; t < MT; t++) {
            if (t >= n) continue;
            const uint8_t *p = qf + (size_t)((unsigned)((tile0 + t) * nb + sb) * (unsigned)FEW_BLOCK);     // (wave-uniform)
#pragma unroll
            for (int s = 0; s < 4; s++) a[t][s] = ldg16(p + s * 1024 + lane * 16);
            const int o = (lane & 15) * 16 + (lane >> 4 & 1) * 8;
            bh[t] = ldg8(p + FEW_BH + o); bl[t] = ldg8(p + FEW_BL + o);
            yd[t] = *reinterpret_cast<const f32x4 *>(p + FEW_D + (lane >> 4) * 16);
        }
    }
};

// the first MT token tiles of A
template <int TYPE, int MT, int M>
__device__ __forceinline__ void superblock(const Frag<TYPE> &R, const Act<M> &A, int kq, bool take, float (*facc)[4]) {
    const i32x4 z = {0, 0, 0, 0};
    if constexpr (Frag<TYPE>::GROUPS) {
        // header: d, dmin, twelve bytes of 6-bit scales and mins
        const uint32_t sc_lo = R.h.y & 0x3f3f3f3fu, mn_lo = R.h.z & 0x3f3f3f3fu;
        const uint32_t sc_hi = (R.h.w & 0x0f0f0f0fu) | ((R.h.y >> 2) & 0x30303030u), mn_hi = ((R.h.w >> 4) & 0x0f0f0f0fu) | ((R.h.z >> 2) & 0x30303030u);
        int isum[MT][4];
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) isum[t][r] = 0;
#define STEP(J)                                                                                              \
        {                                                                                                    \
            const u32x2 b = R.template codes<J>();                                                           \
            const int sc = (int)(((J < 4 ? sc_lo : sc_hi) >> (8 * (J & 3))) & 0xff);                         \
            _Pragma("unroll") for (int t = 0; t < MT; t++) {                                                 \
                const i32x4 I = mfma32((J & 1) ? u32x2{A.a[t][J >> 1].z, A.a[t][J >> 1].w} : u32x2{A.a[t][J >> 1].x, A.a[t][J >> 1].y}, b, z);                                                    \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[t][r] = __mul24(I[r], sc) + isum[t][r];   \
                if constexpr (M > 1) { _Pragma("unroll") for (int r = 0; r < 4; r++) asm volatile("" : "+v"(isum[t][r])); }   /* (the sums are reassociated otherwise, every product alive) */ \
            }                                                                                                \
        }
        STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5) STEP(6) STEP(7)
#undef STEP
        // the mins against the sixteen block sums: min j meets sums 2 j and 2 j + 1; k-quarters 0 and 1 hold them, 2 and 3 are zero
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
            for (int r = 0; r < 4; r++) facc[t][r] += (dd * A.yd[t][r]) * (float)isum[t][r] - (dm * A.yd[t][r]) * (float)ms[r];
        }
    } else {
        // The raw codes against the activations, 16-group by 16-group (a step of 32 weights is two of them: the k-quarters of the other one are
        // zeroed), the signed scale on the four results; the code's "- 32" is the scales against the block sums.  (The scale in the weight, as two int8 planes of
        // sc * (q - 32): 20 instructions per four weights, the head of an 8B model - 431 MB - at 4 tokens 131 us; this form 8 and 16 per token tile: 109 us)
        int isum[MT][4];
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) isum[t][r] = 0;
        const uint32_t m0 = kq < 2 ? ~0u : 0u, m1 = ~m0;
#define STEP(J)                                                                                              \
        {                                                                                                    \
            const u32x2 b = R.template codes<J>();                                                           \
            const uint32_t w = (J >> 1) == 0 ? R.sc.x : (J >> 1) == 1 ? R.sc.y : (J >> 1) == 2 ? R.sc.z : R.sc.w; \
            const int s0 = (int)(int8_t)((w >> (16 * (J & 1))) & 0xff), s1 = (int)(int8_t)((w >> (16 * (J & 1) + 8)) & 0xff); \
            const u32x2 b0 = {b.x & m0, b.y & m0}, b1 = {b.x & m1, b.y & m1};                                \
            _Pragma("unroll") for (int t = 0; t < MT; t++) {                                                 \
                const u32x2 av = (J & 1) ? u32x2{A.a[t][J >> 1].z, A.a[t][J >> 1].w} : u32x2{A.a[t][J >> 1].x, A.a[t][J >> 1].y}; \
                const i32x4 I0 = mfma32(av, b0, z), I1 = mfma32(av, b1, z);                                  \
                _Pragma("unroll") for (int r = 0; r < 4; r++) isum[t][r] = __mul24(I1[r], s1) + (__mul24(I0[r], s0) + isum[t][r]); \
                if constexpr (M > 1 || J == 3) { _Pragma("unroll") for (int r = 0; r < 4; r++) asm volatile("" : "+v"(isum[t][r])); } \
            }                                                                                                \
        }
        STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5) STEP(6) STEP(7)
#undef STEP
        u32x2 bm = kq == 0 ? u32x2{R.sc.x, R.sc.y} : u32x2{R.sc.z, R.sc.w};
        if (kq >= 2) bm = u32x2{0, 0};
        const float dd = h2f((uint16_t)(take ? R.d16 : 0u));
#pragma unroll
        for (int t = 0; t < MT; t++) {
            i32x4 ms = mfma32(A.bh[t], bm, z);
#pragma unroll
            for (int r = 0; r < 4; r++) ms[r] <<= 6;
            ms = mfma32(A.bl[t], bm, ms);
#pragma unroll
            for (int r = 0; r < 4; r++) facc[t][r] += (dd * A.yd[t][r]) * (float)(isum[t][r] - 32 * ms[r]);
        }
    }
}

// LDS of a workgroup: every wave's staging area (NP units), then the sets of partial sums [wave][pair][tile * 4 + r][lane]
template <int TYPE, int NP> constexpr int few_stage = NW * NP * Raw<TYPE == 0 ? T_Q6_K : TYPE>::LDS;
template <int MT, int NP> constexpr int few_sets = MT * NP == 1 ? 2 : 1;  // two in turn: one barrier per tile
template <int TYPE, int MT, int NP> constexpr int few_lds = few_stage<TYPE, NP> + few_sets<MT, NP> * NW * NP * MT * 1024;

// CN > 0: every wave has (up to) CN <= PD super-blocks of a tile and keeps their activation operands in registers across tiles.  CN = 0: any number, the operands
// are read (from the caches) a unit ahead.
// NP = 2: gate and up rows of one SwiGLU pair against the same activation operands.
// HEAD: see mmq_few_head_kernel
constexpr int HEAD_RUN = 4;                                  // row tiles whose results are stored to the host together, a wave's width of rows (two: 16 rows 20 us slower; eight: 4 and 16 rows 8 us)
template <int MT> constexpr int head_lds = 2 * 16 * MT * HEAD_RUN * 64;
template <int TYPE, int MT, int NP, int PD, int CN, bool HEAD = false>
__device__ __forceinline__ void few_body(const FewArgs &a, const MMQSeg &sg, int tile, int n_blocks, uint8_t *smem, int stage_bytes) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, kq = lane >> 4;
    const int nb = a.K >> 8, T = a.T;
    int tiles = (sg.n_rows + 15) >> 4;
    if constexpr (HEAD) {                                    // (a run of neighbours)
        const int b = tile, all = tiles, each = n_blocks;
        tile = (int)((long long)all * b / each); tiles = (int)((long long)all * (b + 1) / each);
        n_blocks = 1;
    }
    const int tile0 = tile;
    uint8_t *stage = smem + wave * (NP * Raw<TYPE>::LDS);
    float *part = reinterpret_cast<float *>(smem + stage_bytes);
    // token tiles are worked on two at a time (the registers of their operands); the operands of a pair that is read again stay a unit ahead
    constexpr int NC = (MT + 1) / 2, PA = CN > 0 ? CN : MT == 1 ? 2 : 1;
    static_assert(CN == 0 || NC == 1, "operands of more than two token tiles are not kept");
    const int cn = CN > 0 ? CN : (nb + NW - 1) / NW;
    float facc[NP][MT][4];
    auto clear = [&]() {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) facc[p][t][r] = 0.0f;
    };
    clear();
    Raw<TYPE> R[PD][NP];
    Act<MT == 1 ? 1 : 2> A[PA][NC];
    // the unit the next request is for; past the end it stays on the last one
    int l_tile = tile, l_i = 0;
    auto request = [&](Raw<TYPE> (&r)[NP]) {
        const int row0 = l_tile * 16, rows = sg.n_rows - row0 < 16 ? sg.n_rows - row0 : 16;
        const int sb = wave + NW * l_i < nb ? wave + NW * l_i : nb - 1;
        r[0].load(sg.W + (size_t)row0 * sg.row_bytes, rows, (unsigned)sg.row_bytes, nb, sb, lane);
        if constexpr (NP == 2) r[1].load(a.seg[1].W + (size_t)row0 * a.seg[1].row_bytes, rows, (unsigned)a.seg[1].row_bytes, nb, sb, lane);
        if (l_i + 1 < cn) l_i++;
        else if (l_tile + n_blocks < tiles) { l_tile += n_blocks; l_i = 0; }
    };
    auto act = [&](Act<MT == 1 ? 1 : 2> &x, int c, int i) {
        const int sb = wave + NW * i;
        x.load(a.qf, blockIdx.y * MT + 2 * c, nb, sb < nb ? sb : nb - 1, lane, MT - 2 * c);
    };
    // an output of a finished tile: element e = tid + NT j of [tile * 4 + r][lane].  Its residual is requested a tile ahead, in front of the weights that follow
    constexpr int NE = (MT * 256 + NT - 1) / NT;
    float rv[NE];
    auto place = [&](int e, int row_tile, size_t &o) {
        const int ln = e & 63, tr = e >> 6;
        const int gt = blockIdx.y * 16 * MT + (tr >> 2) * 16 + 4 * (ln >> 4) + (tr & 3), row = row_tile * 16 + (ln & 15);
        o = (size_t)gt * sg.ld_out + row;
        return e < MT * 256 && gt < T && row < sg.n_rows;
    };
    auto residual = [&](int row_tile) {
        if constexpr (NP == 1) if (sg.resid) {
#pragma unroll
            for (int j = 0; j < NE; j++) { size_t o; const bool in = place(tid + NT * j, row_tile, o); rv[j] = sg.resid[in ? o : 0]; }
        }
    };
    int set = 0;
    // HEAD: results wait in LDS for the other tiles of their run, [run parity][token][row]; a thread's outputs are all of one token
    float *const run = part + few_sets<MT, NP> * NW * NP * MT * 256;
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
        float *ps = part + set * (NW * NP * MT * 256);
        set ^= few_sets<MT, NP> - 1;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) ps[((wave * NP + p) * MT * 4 + t * 4 + r) * 64 + lane] = facc[p][t][r];
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
                    sum += ps[(w * NP) * MT * 256 + e];
                    if constexpr (NP == 2) sum2 += ps[(w * NP + 1) * MT * 256 + e];
                }
                if constexpr (NP == 2) sg.out[o] = (sum / (1.0f + expf(-sum))) * sum2;
                else sg.out[o] = sg.resid ? rv[j] + sum : sum;
                if constexpr (HEAD) {
                    const int k = row_tile - tile0, gt = (e >> 8) * 16 + 4 * ((e & 63) >> 4) + (e >> 6 & 3), row = row_tile * 16 + (e & 15);
                    run[((k / HEAD_RUN & 1) * 16 * MT + gt) * (HEAD_RUN * 16) + (k % HEAD_RUN) * 16 + (e & 15)] = sum;
                    if (sum > top || (sum == top && row < top_row)) { top = sum; top_row = row; }
                }
            }
        }
        if constexpr (few_sets<MT, NP> == 1) __syncthreads();
        clear();
    };
    residual(tile);
#pragma unroll
    for (int i = 0; i < PA; i++)
#pragma unroll
        for (int c = 0; c < NC; c++) act(A[i][c], c, i < cn ? i : 0);
    // (the requests in the order of their use, none moved past another: a wait for one slot must not be a wait for the others)
#pragma unroll
    for (int u = 0; u < PD; u++) { __builtin_amdgcn_sched_barrier(0); request(R[u]); __builtin_amdgcn_sched_barrier(0); }
    static_assert(CN == 0 || PD % CN == 0, "a slot belongs to one super-block of the tile");
    static_assert(CN > 0 || PD % PA == 0, "activation slots turn with the weight slots");
    int i = 0;
    auto unit = [&](Raw<TYPE> (&r)[NP], Act<MT == 1 ? 1 : 2> (&x)[NC], int i) {
        const bool take = wave + NW * i < nb;                              // (a tile of nb super-blocks does not divide by the waves: the last unit's share is multiplied by a zero scale, not branched around)
#pragma unroll
        for (int p = 0; p < NP; p++) r[p].put(stage + p * Raw<TYPE>::LDS, lane);
        uint32_t d16[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) d16[p] = r[p].d16;
        __builtin_amdgcn_sched_barrier(0);                                 // (a wave's LDS accesses are made in order)
        request(r);                                                        // the slot's next unit, in flight across this one's arithmetic
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            constexpr int LAST = MT - 2 * (NC - 1);
#pragma unroll
            for (int p = 0; p < NP; p++) {
                Frag<TYPE> f;
                f.get(stage + p * Raw<TYPE>::LDS, d16[p], n, kq);
                if (c < NC - 1 || LAST == 2) superblock<TYPE, MT == 1 ? 1 : 2>(f, x[c], kq, take, facc[p] + 2 * c);
                else superblock<TYPE, 1>(f, x[c], kq, take, facc[p] + 2 * c);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (CN == 0) { const int j = i + PA; act(x[c], c, j < cn ? j : j - cn < cn ? j - cn : 0); __builtin_amdgcn_sched_barrier(0); }
        }
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
        const int gt = (tid >> 8) * 16 + 4 * (lane >> 4) + (tid >> 6 & 3), blocks = (int)gridDim.x;
        if (tid < MT * 256 && (lane & 15) == 0 && gt < T) {
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
template <int TYPE, int MT, int NP, int PD, int CN>
__global__ __launch_bounds__(NT, 2) void mmq_few_kernel(const FewArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[few_lds<TYPE, MT, NP>];
    int s = 0;
    if constexpr (NP == 1) {
        if (a.n_seg > 1 && (int)blockIdx.x >= a.seg[1].tile0) s = 1;
        if (a.n_seg > 2 && (int)blockIdx.x >= a.seg[2].tile0) s = 2;
    }
    const int first = (int)blockIdx.x - a.seg[s].tile0, n_blocks = (s + 1 < a.n_seg && NP == 1 ? a.seg[s + 1].tile0 : (int)gridDim.x) - a.seg[s].tile0;
    if constexpr (TYPE != 0) few_body<TYPE, MT, NP, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>);
    else switch (a.seg[s].type) {
        case T_Q4_K: few_body<T_Q4_K, MT, NP, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        case T_Q5_K: few_body<T_Q5_K, MT, NP, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        case T_Q6_K: few_body<T_Q6_K, MT, NP, PD, CN>(a, a.seg[s], first, n_blocks, smem, few_stage<TYPE, NP>); break;
        default: break;
    }
}

// The output head of a tick: a workgroup takes a run of neighbouring row tiles, and stores the results of HEAD_RUN of them at a time - 256 consecutive bytes a token - to the
// host's rows while its weights stream: PCIe bounds it from a dozen rows on.  The rows' arg-max is made of what the threads hold anyway.  128256 rows of 4096 columns (Q6_K), us, here /
// the head, the arg-max and a launch that copies the rows one behind the other: 4 tokens 110 / 99 + 10 + 38, 16 tokens 206 / 104 + 19 + 149.
template <int TYPE, int MT, int CN>
__global__ __launch_bounds__(NT, 2) void mmq_few_head_kernel(const FewArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[few_lds<TYPE, MT, 1> + head_lds<MT>];
    few_body<TYPE, MT, 1, 4, CN, true>(a, a.seg[0], (int)blockIdx.x, (int)gridDim.x, smem, few_stage<TYPE, 1>);
}
template <int TYPE>
void few_head(const FewArgs &a, int blocks, hipStream_t st) {
    const int cn = ((a.K >> 8) + NW - 1) / NW;
#define GO(MT, CN) hipLaunchKernelGGL((mmq_few_head_kernel<TYPE, MT, CN>), dim3((unsigned)blocks), dim3(NT), 0, st, a)
    if (a.T <= 16) { if (cn == 1) GO(1, 1); else if (cn == 2) GO(1, 2); else GO(1, 0); }
    else if (cn == 1) GO(2, 1); else if (cn == 2) GO(2, 2); else GO(2, 0);
#undef GO
}

template <int TYPE, int MT, int NP, int PD, int CN>
void few_go(const FewArgs &a, int blocks, hipStream_t st) {
    hipLaunchKernelGGL((mmq_few_kernel<TYPE, MT, NP, PD, CN>), dim3((unsigned)blocks, (unsigned)((a.T + 16 * MT - 1) / (16 * MT))), dim3(NT), 0, st, a);
}
template <int TYPE, int NP>
void few_type(const FewArgs &a, int blocks, hipStream_t st) {
    const int mt = a.T <= 16 ? 1 : a.T <= 32 ? 2 : a.T <= 48 ? 3 : 4, cn = ((a.K >> 8) + NW - 1) / NW;
    constexpr int PD = 4 / NP;                                             // four units of weights in flight per wave: 74 KB per CU
#define GO(MT, CN) few_go<TYPE, MT, NP, PD, CN>(a, blocks, st)
    switch (mt) {
        case 1: if (cn == 1) GO(1, 1); else if (cn == 2) GO(1, 2); else GO(1, 0); break;
        case 2: if (cn == 1) GO(2, 1); else if (cn == 2) GO(2, 2); else GO(2, 0); break;
        case 3: few_go<TYPE, 3, NP, 2 / NP, 0>(a, blocks, st); break;           // (three and four token tiles: their operands take the registers)
        default: few_go<TYPE, 4, NP, 2 / NP, 0>(a, blocks, st); break;
    }
#undef GO
}

}  // namespace

// Whether a launch of T tokens is the faster one here (the sums are the same either way; us, here against the K-split kernel of mmq.hip):
//   * to 16 tokens: 4.2 / 6.1 (2048 x 2048) .. 62 / 100 (128256 x 4096), Q6_K 104 / 139;
//   * to 48: as long as the row tiles fill their rounds of CUs - 320 of 512 do not: 5120 x 5120 14.3 / 10.8 at 17 tokens, 17.9 / 16.4 at 33 - and, for Q6_K, whose units
//     take twice the instructions, there is but one round: 4096 x 4096 10.8 / 13.3, but 6144 x 4096 15.6 / 14.1 and 152064 x 3584 270 / 242;
//   * to 64, where the operands of four token tiles leave two units in flight: gate | up, 42 / 50 (14336 x 4096), and long rows, 32.7 / 39.5 (4096 x 14336) - but 13.5 / 12.7
//     (4096 x 4096), 112 / 77 (8192 x 28672: 512 row tiles), 318 / 217 (152064 x 3584), and Q6_K never, 549 / 233.
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
    // one workgroup per CU where there are more row tiles than that: a segment's share of them by its rows
    const int ns = swiglu ? 1 : n_seg;
    int tiles = 0, type = segs[0].type, blocks = 0;
    for (int i = 0; i < ns; i++) { tiles += (segs[i].n_rows + 15) / 16; if (segs[i].type != type) type = 0; }
    const int cap = std::max(ns, std::min(tiles, num_cu()));
    for (int i = 0, seen = 0; i < n_seg; i++) {
        a.seg[i] = segs[i];
        a.seg[i].tile0 = blocks;
        if (i >= ns) continue;
        seen += (segs[i].n_rows + 15) / 16;
        blocks = std::max(blocks + 1, (int)((long long)cap * seen / tiles));
    }
    if (swiglu) switch (type) {
        case T_Q4_K: few_type<T_Q4_K, 2>(a, blocks, st); break;
        case T_Q5_K: few_type<T_Q5_K, 2>(a, blocks, st); break;
        case T_Q6_K: few_type<T_Q6_K, 2>(a, blocks, st); break;
        default: return hipErrorInvalidValue;
    } else switch (type) {
        case T_Q4_K: few_type<T_Q4_K, 1>(a, blocks, st); break;
        case T_Q5_K: few_type<T_Q5_K, 1>(a, blocks, st); break;
        case T_Q6_K: few_type<T_Q6_K, 1>(a, blocks, st); break;
        default: few_type<0, 1>(a, blocks, st); break;
    }
    return hipGetLastError();
}

static int head_blocks(int n_rows) { return std::min((n_rows + 15) / 16, num_cu()); }
size_t mmq_few_head_scratch() { return 1 + 2 * (size_t)HEAD_MAX_T * (size_t)num_cu(); }
bool mmq_few_head_takes(int type, int K, int T, const ActQuant &q) {
    return q.qf && (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K) && (K & 255) == 0 && T >= 3 && T <= HEAD_MAX_T;
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
