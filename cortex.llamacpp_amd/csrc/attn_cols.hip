// attn_cols.hip — attention of a short batch of one conversation (its next turn, a short prompt) and of a text through the encoder, on the matrix cores.
//
// Scores are the prompt kernel's (attn_prefill.hip: int8 products against q8_0 keys, f16 ones else), the softmax is online in log2 units.  The sums over V are the prompt kernel's for batches
// that it would take, over 64 tokens: weights and q8_0 values as pairs of f16.  Shorter ones come from kernels that hold weights and values in f32, and are no less exact here (EXACT):
// a weight is three f16 parts of 2^15 times itself - with all of f16 below it - and a q8_0 value two, exact from the block's scale and code at any size (pairs of 2^-9 of the values
// where a scale is 512 and more); every product of parts that f32 would see is made.  Error against 64 bits, here with four shares / one-token kernel, geometric mean of 24 conversations at
// 5, 20 and 7 tokens over 100, 700 and 2500 cells, queries of 1 to 10 times unit size: f16 0.81 to 0.94, q8_0 0.88 to 1.01 and with heads of 64 0.96 to 1.04 (as pairs, with one chain of
// eight products for an f16 score: 1.0 to 1.4, and weights under 1e-7 of the largest lost).  It costs 0.3 to 1.2 us a launch.
// The split of the work is another.  What bounds such a call is latency: a kv head's few hundred keys are tens of kilobytes, and a workgroup that stages chunk after chunk in LDS
// for a tile of 32 tokens leaves most of the chip idle behind a chain of barriers.  Here
//   * the columns of a tile are (token, query head of the kv group) pairs, so eight tokens of a 4-heads-per-group model fill one;
//   * a wave takes whole 32-key chunks by itself: K rows ARE the matrix core's A operand and are loaded as such; V rows are loaded four (two) dimensions per lane and
//     key, which makes the lane's dimensions - not 32 consecutive ones - the rows of the output tiles, and needs no transposition.  No staging, no barrier in the loop;
//   * the waves of a workgroup share the tile's keys, the (O, m, l) of each are merged through LDS at the end, and where no other workgroup shares them the merged rows
//     are quantised on the spot: no records, no merge launch.
// Each tile converts V for itself, so a long batch is better off with the prompt kernel (flash_attn_cols_takes).
#include <algorithm>
#include <cstdlib>

#include "kernels.h"
#include "quant_dev.h"

namespace mi355 {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int CK = 32;                                       // keys per chunk, columns per tile
constexpr unsigned V_BIG = 0x6000;                           // f16 512: a block of codes with a smaller scale is within f16

__device__ __forceinline__ float xhalf_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// bytes of a row's DPL dimensions of one lane
template <int B> struct VWord { typedef uint32_t T; };
template <> struct VWord<2> { typedef uint16_t T; };
template <> struct VWord<8> { typedef u32x2 T; };

template <int DH> constexpr int cols_merge_words = (DH / 32) * 16 * 65;      // a wave's O, [16 * tile + register][lane], rows of 65: the readers take registers, not lanes, side by side
template <int DH> constexpr int cols_wave_words = (DH / 32) * CK * 2 + CK + 2 * CK;      // a chunk's scales [k, v][block][key], positions, sequence masks, in the space of the sums
static_assert(cols_wave_words<64> <= cols_merge_words<64> && cols_wave_words<128> <= cols_merge_words<128>, "a chunk's words fit where the wave's sums go");
static_assert(cols_merge_words<64> % 4 == 0 && cols_merge_words<128> % 4 == 0 && CK % 4 == 0, "read 16 and 8 bytes at a time");
template <bool F16, int DH> constexpr int cols_q_stride = (F16 ? 2 * DH : DH) + 16;                            // bytes of a column's query as an operand
template <bool F16, int DH, int NW> constexpr int cols_lds_words = NW * cols_merge_words<DH> + std::max(NW * 64 + CK, CK * cols_q_stride<F16, DH> / 4 + CK * (DH / 32));

struct ColsArgs {
    AttnArgs a;
    ActQuant q;                                              // the merged rows quantised as well (quant: 1 Q8_K, 2 Q8_0); nsp = 1 only
    int quant, nsp, n_chunks;                                // n_chunks: of 32 cells
    float scale_l2;                                          // EXACT: the scores' scale in log2 units, rounded once
    const int32_t *list;                                     // 64-cell chunks to walk (two of 32 each); nullptr: all of [0, n_chunks)
};
static_assert(sizeof(ColsArgs) == 288, "eight bytes more in AttnArgs: 0.2 us a launch at 187 tokens of 12 heads, 0.8 at 65 of 32 / 4");

// EXACT: the products of weights and values as f32 has them (three f16 parts of a weight, a q8_0 value of any size); else as attn_prefill.hip has them
template <bool F16, int DH, int NW, bool EXACT>
__global__ __launch_bounds__(64 * NW, 2) void flash_attn_cols_kernel(const ColsArgs c) {
    constexpr int D = DH, NB = DH / 32, NKS = DH / 16, DPL = DH / 32;
    constexpr float P_ONE = EXACT ? 32768.0f : 1.0f;         // what a weight of one is as an operand: with all of f16 below it
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const AttnArgs &a = c.a;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kg = lane >> 5;
    const int g = blockIdx.x, R = a.H / a.G, n_cols = a.T * R, n_ctx = a.n_ctx;
    int col = blockIdx.y * CK + n;
    const bool q_ok = col < n_cols;
    if (!q_ok) col = n_cols - 1;
    const int tok = col / R, h = g * R + (col - tok * R);
    float *const mine = smem + wave * cols_merge_words<DH>;  // (the chunk's words lie in the space of the wave's own sums)
    float *const s_sc = mine;
    int *const s_pos = reinterpret_cast<int *>(mine + NB * CK * 2);
    unsigned long long *const s_seq = reinterpret_cast<unsigned long long *>(mine + NB * CK * 2 + CK);

    // ---- a chunk as it is requested: K rows as the A operand (row n = key), V words of key slots (j, kg, i), scales and cell data of key `lane & 31`
    typedef typename VWord<F16 ? 2 * DPL : DPL>::T vword;
    i32x4 kq[F16 ? NKS : NB];
    vword vq[2][8];
    uint32_t sq[2];
    int cp;
    unsigned long long cs;
    int n_kv;
    auto cell_of = [&](int i) { return c.list ? (c.list[i >> 1] << 6) + ((i & 1) << 5) : i << 5; };
    // a head's rows by 32-bit offsets from a scalar base (a 64-bit address per row and lane takes the registers of everything else)
    constexpr unsigned RB = F16 ? 2 * D : D;
    const uint8_t *const kb = a.kv.k + (size_t)g * n_ctx * RB, *const vb = a.kv.v + (size_t)g * n_ctx * RB;
    const uint8_t *const kdb = (const uint8_t *)(a.kv.kd + (size_t)g * n_ctx * NB), *const vdb = (const uint8_t *)(a.kv.vd + (size_t)g * n_ctx * NB);
    const auto row_of = [&](int cell0, int key) { const int x = cell0 + key; return (unsigned)(x < n_ctx ? x : n_ctx - 1); };
    auto load_k = [&](int i) {                               // ... and what belongs to the keys
        const int cell0 = cell_of(i);
        const unsigned kr = row_of(cell0, n) * RB + 16u * kg;
#pragma unroll
        for (int j = 0; j < (F16 ? NKS : NB); j++) kq[j] = *reinterpret_cast<const i32x4 *>(kb + kr + 32 * j);
        if constexpr (!F16) {
            const unsigned so = row_of(cell0, n) * (2 * NB);
            if constexpr (NB == 4) { const u32x2 x = kg ? *reinterpret_cast<const u32x2 *>(vdb + so) : *reinterpret_cast<const u32x2 *>(kdb + so); sq[0] = x.x; sq[1] = x.y; }
            else sq[0] = kg ? *reinterpret_cast<const uint32_t *>(vdb + so) : *reinterpret_cast<const uint32_t *>(kdb + so);
        }
        const unsigned cc = row_of(cell0, n);
        cp = a.cell_pos[cc]; cs = a.cell_seq[cc];
        if (cell0 + n >= n_ctx) cp = -1;
    };
    auto load_v = [&](int i) {
        const int cell0 = cell_of(i);
        unsigned o = 0;
        asm volatile("" : "+v"(o));                          // (the offsets are formed here, every time)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i2 = 0; i2 < 8; i2++)
                vq[j][i2] = *reinterpret_cast<const vword *>(vb + (row_of(cell0, 16 * j + 8 * (i2 >> 2) + 4 * kg + (i2 & 3)) * RB + (n * (unsigned)sizeof(vword) + o)));
    };
    const int first = (int)blockIdx.z * NW + wave, step = c.nsp * NW;
    if (first < c.n_chunks) { load_k(first); load_v(first); }
    const int tpos = a.tok_pos[tok], tseq = a.tok_seq[tok];
    n_kv = *a.n_kv_dev;

    // ---- the tile's queries, quantised by all waves: Q8_0 blocks as flash_attn_ext quantises them (f16 cache: rounded to f16)
    uint8_t *const s_q = reinterpret_cast<uint8_t *>(smem + NW * cols_merge_words<DH>);       // [column][D], behind them the block scales [column][block]
    float *const s_dq = smem + NW * cols_merge_words<DH> + CK * cols_q_stride<F16, DH> / 4;
    constexpr int QS = cols_q_stride<F16, DH>;
    {
        constexpr int EPT = CK * D / (64 * NW), TPB = 32 / EPT;          // a thread's elements, threads of a 32-block
        static_assert(EPT >= 4 && EPT <= 16 && TPB >= 2 && TPB <= 8, "a block within eight lanes");
        const int e0 = tid * EPT, cl = e0 / D, d0 = e0 - cl * D;
        const int qc = blockIdx.y * CK + cl < n_cols ? blockIdx.y * CK + cl : n_cols - 1, qt = qc / R, qhd = g * R + (qc - qt * R);
        const float *src = a.q + ((size_t)qt * a.H + qhd) * D + d0;
        f32x4 x[EPT / 4];
#pragma unroll
        for (int i = 0; i < EPT / 4; i++) x[i] = *reinterpret_cast<const f32x4 *>(src + 4 * i);
        if constexpr (F16) {
#pragma unroll
            for (int i = 0; i < EPT / 4; i++) {
                typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<f16x4 *>(s_q + cl * QS + 2 * (d0 + 4 * i)) = f16x4{(_Float16)x[i].x, (_Float16)x[i].y, (_Float16)x[i].z, (_Float16)x[i].w};
            }
        } else {
            float am = 0.0f;
#pragma unroll
            for (int i = 0; i < EPT / 4; i++) am = fmaxf(am, fmaxf(fmaxf(fabsf(x[i].x), fabsf(x[i].y)), fmaxf(fabsf(x[i].z), fabsf(x[i].w))));
            am = fmaxf(am, dpp_f<DPP_QP_1032>(am));
            if constexpr (TPB >= 4) am = fmaxf(am, dpp_f<DPP_QP_2301>(am));
            if constexpr (TPB >= 8) am = fmaxf(am, dpp_f<DPP_HALF_MIRROR>(am));
            const float d = am / 127.0f;
            const float id = d != 0.0f ? 1.0f / d : 0.0f;
#pragma unroll
            for (int i = 0; i < EPT / 4; i++) {
                const int c0 = (int)roundf(x[i].x * id), c1 = (int)roundf(x[i].y * id), c2 = (int)roundf(x[i].z * id), c3 = (int)roundf(x[i].w * id);
                *reinterpret_cast<uint32_t *>(s_q + cl * QS + d0 + 4 * i) = (uint32_t)((c0 & 0xff) | ((c1 & 0xff) << 8) | ((c2 & 0xff) << 16) | ((c3 & 0xff) << 24));
            }
            if (tid % TPB == 0) s_dq[cl * NB + (d0 >> 5)] = h2f(f2h(d));
        }
    }
    // ---- what the tile's columns can see (both halves of the wave hold the same columns)
    int maxpos, minpos;
    unsigned long long seqs;
    {
        int hi = tpos, lo = tpos;
#define ACROSS(CTRL) { hi = max(hi, dpp_i<CTRL>(hi)); lo = min(lo, dpp_i<CTRL>(lo)); }
        ACROSS(DPP_QP_1032) ACROSS(DPP_QP_2301) ACROSS(DPP_HALF_MIRROR) ACROSS(DPP_MIRROR)
#undef ACROSS
        maxpos = max(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(hi, 16));
        minpos = min(__builtin_amdgcn_readlane(lo, 0), __builtin_amdgcn_readlane(lo, 16));
        seqs = 0ull;
        for (unsigned long long left = __ballot(true); left;) {         // (a turn per sequence: mostly one)
            const int sq0 = __builtin_amdgcn_readlane(tseq, __builtin_ctzll(left));
            seqs |= 1ull << sq0;
            left &= ~__ballot(tseq == sq0);
        }
    }
    __syncthreads();
    i32x4 qc[F16 ? 1 : NB];
    float dq[F16 ? 1 : NB];
    f16x8 qh[F16 ? NKS : 1];
    if constexpr (F16) {
#pragma unroll
        for (int j = 0; j < NKS; j++) qh[j] = *reinterpret_cast<const f16x8 *>(s_q + n * QS + (16 * j + 8 * kg) * 2);
    } else {
#pragma unroll
        for (int b = 0; b < NB; b++) { qc[b] = *reinterpret_cast<const i32x4 *>(s_q + n * QS + 32 * b + 16 * kg); dq[b] = s_dq[n * NB + b]; }
    }
    const bool one = (seqs & (seqs - 1)) == 0ull;            // (then a cell of another sequence is hidden like an empty one)
    float m_run = -INFINITY, l_run = 0.0f;
    const float scale_l2 = EXACT ? c.scale_l2 : a.scale * 1.4426950408889634f;
    f32x16 O[NB];                                            // P_ONE times the sums
#pragma unroll
    for (int db = 0; db < NB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) O[db][r] = 0.0f;

    for (int ci = first; ci < c.n_chunks; ci += step) {
        // the chunk's scales and cells through LDS (the wave's own); the next chunk's K rows are requested behind the scores, its V rows behind P . V
        const int cell = cell_of(ci) + n;
        const bool live = cell < n_kv && cp >= 0 && cp <= maxpos && (cs & seqs) != 0ull;
        const bool open = __all(cell < n_kv && cp >= 0 && cp <= minpos && (cs & seqs) == seqs);
        const bool more = ci + step < c.n_chunks, see = __any(live);     // (wave-uniform)
        bool big = false;                                    // a value of the chunk may be beyond f16
        if constexpr (EXACT && !F16) {
            unsigned top = 0;
#pragma unroll
            for (int b = 0; b < NB; b++) top = max(top, (sq[b >> 1] >> (16 * (b & 1))) & 0x7fffu);
            big = __any(kg == 1 && top >= V_BIG);
        }
        if (kg == 0) { s_pos[n] = live ? cp : -1; if (!one) s_seq[n] = cs; }
        if constexpr (!F16) {
#pragma unroll
            for (int b = 0; b < NB; b++) s_sc[(kg * NB + b) * CK + n] = h2f((uint16_t)(sq[b >> 1] >> (16 * (b & 1))));
        }
        asm volatile("" ::: "memory");                       // (a wave's LDS accesses are made in order)
        float sc[16];
        if (see) {
        if constexpr (F16) {
            constexpr int CH = EXACT ? 2 : 1;                 // (sums of half of the dimensions each: a chain of eight loses more than the one-token kernel's)
            f32x16 sa[CH];
#pragma unroll
            for (int k = 0; k < CH; k++)
#pragma unroll
                for (int r = 0; r < 16; r++) sa[k][r] = 0.0f;
#pragma unroll
            for (int j = 0; j < NKS; j++) sa[j * CH / NKS] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, kq[j]), qh[j], sa[j * CH / NKS], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = CH > 1 ? sa[0][r] + sa[CH - 1][r] : sa[0][r];
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = 0.0f;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                i32x16 z;
#pragma unroll
                for (int r = 0; r < 16; r++) z[r] = 0;
                const i32x16 I = __builtin_amdgcn_mfma_i32_32x32x32_i8(kq[b], qc[b], z, 0, 0, 0);
                if (b & 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rq = 0; rq < 4; rq++) {
                    const f32x4 dk4 = *reinterpret_cast<const f32x4 *>(s_sc + b * CK + 8 * rq + 4 * kg);
#pragma unroll
                    for (int ri = 0; ri < 4; ri++) sc[rq * 4 + ri] += (float)I[rq * 4 + ri] * (dq[b] * dk4[ri]);
                }
            }
        }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_k(ci + step);
        __builtin_amdgcn_sched_barrier(0);
        if (see) {
        float mloc = -INFINITY;
        if (open) {
#pragma unroll
            for (int r = 0; r < 16; r++) { if constexpr (!EXACT) sc[r] *= scale_l2; mloc = fmaxf(mloc, sc[r]); }
        } else {
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const i32x4 kp = *reinterpret_cast<const i32x4 *>(s_pos + 8 * rq + 4 * kg);
#pragma unroll
                for (int ri = 0; ri < 4; ri++) {
                    const int r = 4 * rq + ri;
                    bool vis = (unsigned)kp[ri] <= (unsigned)tpos;       // (-1: hidden from all)
                    if (!one) vis = vis & ((s_seq[8 * rq + 4 * kg + ri] >> tseq & 1ull) != 0ull);
                    sc[r] = vis ? EXACT ? sc[r] : sc[r] * scale_l2 : -INFINITY;
                    mloc = fmaxf(mloc, sc[r]);
                }
            }
        }
        mloc = xhalf_max(mloc);
        if constexpr (EXACT) mloc *= scale_l2;
        const float m_new = fmaxf(m_run, mloc);
        const float m_ref = m_new == -INFINITY ? 0.0f : m_new;
        float p[16], lsum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) { p[r] = __builtin_amdgcn_exp2f(EXACT ? __builtin_fmaf(sc[r], scale_l2, -m_ref) : sc[r] - m_ref); if constexpr (!EXACT) lsum += p[r]; }
        if constexpr (EXACT) {                               // (in pairs: what the sum loses is every dimension's loss)
            float t[8];
#pragma unroll
            for (int r = 0; r < 8; r++) t[r] = p[2 * r] + p[2 * r + 1];
            lsum = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
        }
        lsum = xhalf_sum(lsum);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
        l_run = EXACT ? __builtin_fmaf(l_run, alpha, lsum) : l_run * alpha + lsum;
        m_run = m_new;
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int db = 0; db < NB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) O[db][r] *= alpha;
        }
        // (a chunk whose values may be beyond f16 is added in two turns, the larger values as 2^-9 of theirs)
#pragma unroll 1
        for (int turn = 0; turn <= (int)big; turn++) {
            if (turn) {
#pragma unroll
                for (int db = 0; db < NB; db++)
#pragma unroll
                    for (int r = 0; r < 16; r++) O[db][r] *= 0x1p-9f;
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                f16x8 ph, pm, pl;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if constexpr (EXACT && !F16) asm volatile("" : "+v"(p[8 * j + i]), "+v"(vq[j][i]));        // (nothing made of them is kept from turn to turn)
                    const float v = EXACT ? p[8 * j + i] * P_ONE : p[8 * j + i];
                    ph[i] = (_Float16)v;
                    const float w = v - (float)ph[i];
                    pm[i] = (_Float16)w;
                    if constexpr (EXACT) pl[i] = (_Float16)(w - (float)pm[i]);
                }
                // output tile db, row m: dimension DPL m + db
                if constexpr (F16) {
#pragma unroll
                    for (int db = 0; db < NB; db++) {
                        u32x4 w;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            uint32_t lo, hi;
                            if constexpr (DPL == 4) { lo = vq[j][2 * i][db >> 1]; hi = vq[j][2 * i + 1][db >> 1]; }
                            else { lo = vq[j][2 * i]; hi = vq[j][2 * i + 1]; }
                            w[i] = __builtin_amdgcn_perm(hi, lo, (db & 1) ? 0x07060302u : 0x05040100u);
                        }
                        const f16x8 av = __builtin_bit_cast(f16x8, w);
                        if constexpr (EXACT) {
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, pl, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, pm, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, ph, O[db], 0, 0, 0);
                        } else {
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, ph, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, pm, O[db], 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    float dv[8];
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const f32x4 x = *reinterpret_cast<const f32x4 *>(s_sc + (NB + ((DPL * n) >> 5)) * CK + 16 * j + 8 * q + 4 * kg);
#pragma unroll
                        for (int e = 0; e < 4; e++) dv[4 * q + e] = x[e];
                    }
                    if (big) {
#pragma unroll
                        for (int i = 0; i < 8; i++) { const bool small = fabsf(dv[i]) < 512.0f; dv[i] = turn ? small ? 0.0f : dv[i] * 0x1p-9f : small ? dv[i] : 0.0f; }
                    }
#pragma unroll
                    for (int db = 0; db < NB; db++) {
                        f16x8 vh, vl;
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            const float v = (float)(int8_t)((vq[j][i] >> (8 * db)) & 0xff) * dv[i];
                            vh[i] = (_Float16)v;
                            vl[i] = (_Float16)(v - (float)vh[i]);
                        }
                        if constexpr (EXACT) {               // (the small ones first: the other way round q8_0 is up to 0.1 further off)
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, pm, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pm, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph, O[db], 0, 0, 0);
                        } else {
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pm, O[db], 0, 0, 0);
                            O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph, O[db], 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            if (turn) {
#pragma unroll
                for (int db = 0; db < NB; db++)
#pragma unroll
                    for (int r = 0; r < 16; r++) O[db][r] *= 0x1p9f;
            }
        }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_v(ci + step);
        asm volatile("" ::: "memory");
    }

    // ---- the waves' shares as softmax partials over disjoint keys: O = sum_w O_w 2^(m_w - m)
    float *const s_ml = smem + NW * cols_merge_words<DH>;    // [wave][m, l][column], where the queries were
    __syncthreads();
    if (kg == 0) { s_ml[wave * 64 + n] = m_run; s_ml[wave * 64 + 32 + n] = l_run; }
    __syncthreads();
    float m_all = -INFINITY, l_all = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) m_all = fmaxf(m_all, s_ml[w * 64 + n]);
    const float m_ref = m_all == -INFINITY ? 0.0f : m_all;
#pragma unroll
    for (int w = 0; w < NW; w++) l_all += s_ml[w * 64 + 32 + n] * __builtin_amdgcn_exp2f(s_ml[w * 64 + n] - m_ref);
    // (the merge of the shares works in natural-log units: what the record's maximum loses by its rounding goes into the sums)
    const float m_nat = m_all * 0.6931471805599453f;
    const float adj = EXACT && c.nsp > 1 && m_all != -INFINITY ? __builtin_amdgcn_exp2f(__builtin_fmaf(-m_nat, 1.925963033500e-08f, __builtin_fmaf(-m_nat, 1.44269502162933349609375f, m_all))) : 1.0f;
    const float f = __builtin_amdgcn_exp2f(m_run - m_ref) * (adj * (1.0f / P_ONE));
    float *const s_l = s_ml + NW * 64;                       // (a column's sum, for the end)
    if (wave == 0 && kg == 0) s_l[n] = l_all;
#pragma unroll
    for (int db = 0; db < NB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) mine[(db * 16 + r) * 65 + lane] = O[db][r] * f;
    if (wave == 0 && kg == 0 && c.nsp > 1 && q_ok) {
        float *rec = a.part + (((size_t)tok * a.H + h) * c.nsp + blockIdx.z) * att_rec(D);
        rec[D] = m_nat; rec[D + 1] = l_all * adj;
    }
    __syncthreads();
    // a wave per 256 values: 256 / D columns, four consecutive dimensions per lane
    constexpr int CPB = 256 / D, LPC = D / 4;
    const int cw = lane / LPC, d0 = (lane - cw * LPC) * 4;
    for (int b = wave; b < CK / CPB; b += NW) {
        const int cb = b * CPB + cw, gc = blockIdx.y * CK + cb;
        const float l = c.nsp > 1 ? 1.0f : s_l[cb];          // (divided by once, behind the sum over the waves)
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int d = d0 + e, m = d / DPL, db = d - m * DPL, r = (m & 3) + 4 * (m >> 3), o = (db * 16 + r) * 65 + cb + 32 * ((m >> 2) & 1);
            float x[NW];                                     // (in pairs: three roundings instead of seven)
#pragma unroll
            for (int w = 0; w < NW; w++) x[w] = smem[w * cols_merge_words<DH> + o];
#pragma unroll
            for (int h = NW / 2; h >= 1; h >>= 1)
#pragma unroll
                for (int w = 0; w < h; w++) x[w] += x[w + h];
            v[e] = x[0] / l;
        }
        if (blockIdx.y * CK + b * CPB >= n_cols) break;      // (wave-uniform)
        const bool in = gc < n_cols;
        const int t = in ? gc / R : 0, hh = g * R + (gc - t * R);
        if (c.nsp > 1) {
            if (in) {
                float *rec = a.part + (((size_t)t * a.H + hh) * c.nsp + blockIdx.z) * att_rec(D) + d0;
                *reinterpret_cast<f32x2 *>(rec) = f32x2{v[0], v[1]}; *reinterpret_cast<f32x2 *>(rec + 2) = f32x2{v[2], v[3]};
            }
            continue;
        }
        if (in) *reinterpret_cast<f32x4 *>(a.out + ((size_t)t * a.H + hh) * D + d0) = f32x4{v[0], v[1], v[2], v[3]};
        if (c.quant) {                                       // (the columns of a block are then whole: cols_quantises)
            const int E = a.H * D, blk = (hh * D) >> 8;
            if (c.quant & 1) {
                uint32_t packed; int bs; float dqv;
                wave_quant_q8k(v, lane, packed, bs, dqv);
                store_q8k(c.q, t, E, blk, lane, packed, bs, dqv, a.out_bh, a.out_bl);
            }
            if (c.quant & 2) {
                uint32_t packed; float dd;
                wave_quant_q80(v, packed, dd);
                const size_t e0 = (size_t)t * E + hh * D + d0;
                *reinterpret_cast<uint32_t *>(c.q.qs0 + e0) = packed;
                if ((lane & 7) == 0) c.q.d0[e0 >> 5] = f2h(dd);
            }
        }
    }
}

// a block of 256 output values is 256 / D consecutive columns of one token
bool cols_quantises(const AttnArgs &a) {
    const int R = a.H / a.G;
    return (R * a.D) % 256 == 0;
}

}  // namespace

static int cols_chunks(const AttnArgs &a) { return a.chunks ? 2 * a.n_chunks : (std::min(a.n_kv_max, a.n_ctx) + CK - 1) / CK; }
static int cols_tiles(const AttnArgs &a) { return a.G * ((a.T * (a.H / a.G) + CK - 1) / CK); }
// How many workgroups share a tile's keys.  A workgroup fills a CU; of its time (us, as the tables below have it) a part is its start and its end, the rest goes by the rounds
// of chunks that its waves walk, and sharing costs the records and the launch that merges them.  Four waves where a share is no more than four chunks.  Measured (us, attention and merge, weights
// as pairs; EXACT adds 0.3 to 1.2):
//   32 / 8 heads of 128, q8_0      37 tokens, 677 cells: 1 share 19.8, 2 19.8, 3 15.1, 6 15.0, 12 15.9      64, 677: 20.1, 20.4, 16.0, 18.5, 21.0
//                                  37, 3900: 1 71.7, 3 34.4, 6 26.3, 8 36.0, 16 38.6                        5, 3900: 1 70.3, 6 21.9, 16 13.8, 32 13.4
//   32 / 4 heads of 64, f16        37, 677: 1 11.4, 3 12.3, 6 12.8                                          2, 677: 1 10.5, 3 9.4, 6 8.2
// The tiles are those of the caller's kv heads: a rank of a row split, with a part of them, shares its keys in another number of parts than the whole model does, and its sums differ from the
// whole's by the order of f32 additions - as its attn_output and ffn_down, summed over the ranks, do anyway.  Greedy answers of a split model can part from the unsplit one's at a near tie.
static double cols_time(const AttnArgs &a, int nsp) {
    const int per = (cols_chunks(a) + nsp - 1) / nsp, nw = per > 4 ? 8 : 4, walks = (per + nw - 1) / nw, rounds = (cols_tiles(a) * nsp + num_cu() - 1) / num_cu();
    const double start = a.D == 128 ? 6.5 : 5.0, walk = a.D == 128 ? 4.0 : 2.1, merge = 2.5 + 2.5 * std::min(a.T, 32) / 32;
    return rounds * (start - (nw == 4 ? 1.0 : 0.0) + walk * walks) + (nsp > 1 ? merge : 0.0);
}
int flash_attn_cols_splits(const AttnArgs &a) {
    int best = 1;
    for (int n = 2; n <= std::min(64, (cols_chunks(a) + 3) / 4); n++) if (cols_time(a, n) < cols_time(a, best)) best = n;
    return best;
}

bool flash_attn_cols_applicable(const AttnArgs &a) {
    if (a.G < 1 || a.H % a.G != 0 || (a.D != 64 && a.D != 128) || a.T < 1 || a.n_kv_max < 1) return false;
    const bool f16 = a.type_k == T_F16 && a.type_v == T_F16, q8 = a.type_k == T_Q8_0 && a.type_v == T_Q8_0;
    return (f16 || q8) && (int64_t)a.T * (a.H / a.G) <= (65535LL * CK) && (a.H * a.D) % 256 == 0;
}

// Long batches, here / attn_prefill.hip with its merge (us a layer):
//   32 / 8 heads of 128, q8_0   64 tokens behind 613 cells 18 / 39, 256 / 0 15 / 29, 256 / 3500 88 / 98, 450 / 3400 163 / 195, 512 / 0 34 / 44, 512 / 1500 101 / 102, 512 / 2488 145 / 137,
//                               512 / 3400 169 / 161
//   32 / 32 heads of 128, f16   256 / 2000 53 / 63, 300 / 2000 85 / 103, 512 / 0 28 / 41, 512 / 1000 67 / 69, 512 / 1500 86 / 83, 400 / 2500 113 / 101, 450 / 1500 82 / 77, 512 / 2500 122 / 109
//   32 / 4 heads of 64, f16     256 / 0 8 / 24, 768 / 1200 66 / 80, 850 / 0 44 / 45, 1024 / 0 51 / 50, 1024 / 900 86 / 75      12 / 12 heads of 64, f16 (a text)   187 6.6 / 17, 2000 58 / 92
// (These are the prompt kernel's with every tile converting V for itself.  With the planes made once a layer it is ahead at 512 / 1000 and 512 / 1400 q8_0 by 8 and 10 us a layer and at 450 / 3400 by
// 4, behind at 512 / 0, 350 / 3500, 256 / 2000 by 10, 10 and 7 and at 300 / 2000 f16 by 20: one to two hundredths of a pass on either side of a line, which stays.)
// So with heads of 64 three rounds of workgroups; with heads of 128 two as long as the keys are few, to 1536 cells with a query head to every kv head and to 2048 else, and with more keys
// 11 / 8 and 15 / 8 rounds.
static bool cols_long(const AttnArgs &a) {
    const int eighths = 8 * cols_tiles(a), cu = num_cu(), ch = cols_chunks(a);
    if (a.D == 64) return eighths <= 24 * cu;
    return eighths <= (a.H == a.G ? ch <= 48 ? 16 : 11 : ch <= 64 ? 16 : 15) * cu;
}
// Short ones beside the one-token kernel, a (token, 64-cell chunk) at a time with a merge, whose sums are a step's: here / there, T tokens behind so many cells, each with its merge
//   32 / 8 heads of 128, q8_0   2 / 2100 13.2 / 13.6, 3 / 1900 14.1 / 14.7, 5 / 900 14.1 / 12.9, 5 / 1495 14.8 / 15.7, 8 / 700 14.2 / 13.3, 12 / 400 14.3 / 12.6, 14 / 700 14.7 / 17.3,
//                               22 / 200 13.3 / 12.6, 31 / 150 13.7 / 12.9, 31 / 200 13.1 / 14.6, 32 / 0 11.4 / 10.8, 40 / 0 11.3 / 11.2, 64 / 0 11.0 / 11.4
//   32 / 32 heads of 128, f16   2 / 2100 20.4 / 17.0, 2 / 3000 21.2 / 24.0, 2 / 3900 22 / 29, 3 / 1900 17.0 / 19.2, 5 / 900 13.5 / 16.8, 12 / 400 12.3 / 16.5, 32 / 0 8.3 / 10.7
//   32 / 4 heads of 64, f16     3 / 1900 11.7 / 15.6, 8 / 700 10.1 / 14.6, 22 / 200 7.4 / 14.4
// A pass of eight layers with heads of 128, us, at 2, 4, 8, 16 and 31 tokens, here / there, behind so many cells:
//   32 / 32, f16     0  770 / 783, 606 / 618, 618 / 637, 652 / 669, 761 / 783     200  792 / 788, 642 / 632, 663 / 672     260  787 / 792, 631 / 635, 639 / 654     500  789 / 791, 619 / 635, 641 / 664
//   32 / 8, f16      0  749 / 772, 648 / 652, 658 / 667, 674 / 685, 762 / 777     330  775 / 763, 668 / 653, 682 / 667, 697 / 702
//   32 / 8, q8_0     20  761 / 781, 648 / 650, 666 / 664, 694 / 688     90  751 / 765, 643 / 652, 671 / 667, 689 / 691     130  768 / 770, 661 / 659, 680 / 669
// So here while the cells are two chunks of 64, a q8_0 cache's to four tokens, and for f16 heads with keys of their own from four tokens and five chunks on; else by the work.
// Where no store of K and V goes with the one-token kernel (fewer than 1024 values a row, NEOX pairs), the general attention is what there is, which knows no lists and needs a merge: here
// at any size.  (Within one chunk of cells and heads of 64, 2 to 31 tokens, the attention alone is 1.2e-7 to 1.35e-7 from 64 bits here and 1.5e-7 to 1.6e-7 there with an f16 cache, 1.1e-7 to 1.25e-7 and 1.2e-7 to
// 1.3e-7 with a q8_0 one.)  A pass, us, at 2, 3, 8, 16 and 31 tokens, here / there:
//   six layers, 32 / 4 of 64, f16           0  327 / 365, 371 / 414, 370 / 415, 376 / 425, 383 / 437     200  347 / 391, 397 / 452, 389 / 438     1500  355 / 387, 396 / 440
//   32 / 8 of 64, f16                       0  337 / 365, 375 / 406, 374 / 408, 379 / 410, 387 / 433     330  368 / 382, 412 / 434, 405 / 434
//   four layers, 28 / 4 of 128, NEOX, q8_0  0  362 / 364, 358 / 362, 372 / 388, 383 / 406, 437 / 480     130  366 / 407, 365 / 404, 377 / 414, 386 / 433, 443 / 502     1500  371 / 412, 367 / 415      f16 130  349 / 392, 353 / 392, 361 / 402, 375 / 420
//   six layers, 12 / 2 of 128, NEOX, f16    130  404 / 458, 360 / 413, 369 / 407, 378 / 415, 407 / 413     900  394 / 440, 345 / 379
// (Nor has the encoder a one-token kernel: 3 tokens 5.7 / 7.9 with the general one.)
static bool cols_short(const AttnArgs &a) {
    const int ch = (cols_chunks(a) + 1) / 2, work = a.T * ch;
    const bool wide = a.D == 128, q8 = a.type_k == T_Q8_0;
    if (a.T >= (wide && q8 ? 40 : 32)) return true;
    if (wide && ch <= 2 && (!q8 || a.T <= 4)) return true;
    if (wide && !q8 && a.H == a.G && ch >= 5 && a.T >= 4) return true;
    return work >= (!wide ? 64 : q8 ? ch < 28 ? 104 : 64 : a.T < 3 ? 80 : 64);
}
bool flash_attn_cols_takes(const AttnArgs &a, bool one_token_kernel) {
    static const bool off = getenv("MI355_ATTN_COLS") && getenv("MI355_ATTN_COLS")[0] == '0';
    return !off && flash_attn_cols_applicable(a) && cols_long(a) && (!one_token_kernel || cols_short(a));
}

template <bool F16, int DH, int NW, bool EXACT>
static void cols_go(const ColsArgs &c, hipStream_t st) {
    const AttnArgs &a = c.a;
    constexpr int lds = cols_lds_words<F16, DH, NW> * 4;
    if (lds > 65536) (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&flash_attn_cols_kernel<F16, DH, NW, EXACT>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL((flash_attn_cols_kernel<F16, DH, NW, EXACT>), dim3((unsigned)a.G, (unsigned)(cols_tiles(a) / a.G), (unsigned)c.nsp), dim3(64 * NW), lds, st, c);
}

hipError_t launch_flash_attn_cols(const AttnArgs &a, hipStream_t st) {
    if (!flash_attn_cols_applicable(a)) return hipErrorInvalidValue;
    ColsArgs c{};
    c.a = a;
    c.nsp = a.pf_splits > 1 && a.part ? a.pf_splits : 1;
    c.scale_l2 = (float)((double)a.scale * 1.4426950408889634);
    c.n_chunks = cols_chunks(a);
    c.list = a.chunks;
    const bool here = c.nsp == 1 && a.out_q && cols_quantises(a);
    if (here) { c.q = act_for(a.out_q, a.T); c.quant = (a.out_q8k ? 1 : 0) | (a.out_q80 ? 2 : 0); }
    const bool wide = c.n_chunks > 4 * c.nsp;
    const bool exact = a.T <= 64 || !flash_attn_prefill_applicable(a);
#define GO1(F, DD, X) do { if (wide) cols_go<F, DD, 8, X>(c, st); else cols_go<F, DD, 4, X>(c, st); } while (0)
#define GO(F, DD) do { if (exact) GO1(F, DD, true); else GO1(F, DD, false); } while (0)
    if (a.type_k == T_F16) { if (a.D == 128) GO(true, 128); else GO(true, 64); }
    else if (a.D == 128) GO(false, 128);
    else GO(false, 64);
#undef GO
#undef GO1
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (c.nsp > 1) return launch_flash_attn_combine(a, c.nsp, st);
    if (a.out_q && !here) e = launch_quantize(a.out, a.H * a.D, a.T, *a.out_q, a.out_q8k, a.out_q80, st, a.out_bh, a.out_bl);
    return e;
}

}  // namespace mi355
