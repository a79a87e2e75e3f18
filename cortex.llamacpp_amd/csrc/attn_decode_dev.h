// attn_decode_dev.h — device side of the decode attention (one 64-cell chunk of one kv head per 256-thread workgroup).
// Shared by attn.hip (one launch per layer) and decode_mega.hip (a phase of the whole-step kernel).
#pragma once
#include <type_traits>

#include "kernels.h"
#include "quant_dev.h"

namespace mi355 {

// quantize_row_q4_0 of a 32-block held by 8 consecutive lanes, 4 consecutive values each: the FIRST element of largest magnitude sets d = max / -8, codes
// min(15, (int8)(x / d + 8.5)); nib4 = this lane's four codes, one per byte (0 .. 15).  The block's 16 bytes are q[j] | q[j + 16] << 4: lanes 0-3 of the group
// hold the low nibbles, lanes 4-7 the high ones (combine with the lane 4 further on).
__device__ __forceinline__ void wave_quant_q40(const float (&vv)[4], int lane, uint32_t &nib4, float &d) {
    // key: |x| bits above, first-index preference below (larger key = larger magnitude, then smaller index)
    unsigned long long key = 0ull;
    float vbest = 0.0f;
#pragma unroll
    for (int i = 3; i >= 0; i--) {
        const unsigned long long k = ((unsigned long long)__float_as_uint(fabsf(vv[i])) << 32) | (unsigned long long)(0xffffffffu - (unsigned)((lane & 7) * 4 + i));
        if (k > key) { key = k; vbest = vv[i]; }
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        const unsigned long long ok = __shfl_xor(key, o, 64);
        const float ov = __shfl_xor(vbest, o, 64);
        if (ok > key) { key = ok; vbest = ov; }
    }
    d = vbest / -8.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    nib4 = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int q = (int)(int8_t)(vv[i] * id + 8.5f);
        q = q > 15 ? 15 : q;
        nib4 |= (uint32_t)(q & 0xff) << (8 * i);
    }
}

// four nibbles (one per byte, 0 .. 15) -> the int8 codes nibble - 8, per byte without borrows across bytes
__device__ __forceinline__ uint32_t nib_to_i8x4(uint32_t n) { return ((n | 0x80808080u) - 0x08080808u) ^ 0x80808080u; }

// Decode attention: workgroup = (kv head g, chunk of 64 cells, token t).  The query heads of the group are read
// un-rotated, rotated with the cos/sin table and converted to the K cache's dot type here (so no separate pass over q),
// and K / V / scales / cell table of the chunk are all requested before the first wait.
//
// FUSED (single-token step, R*D a multiple of 256) folds the two neighbouring launches into this one:
//  * KV store: the workgroup whose chunk holds the token's cell rotates K, converts K/V to the cache type, writes the
//    cache row and patches its own registers / LDS scales with the same codes (no other workgroup reads that cell).
//    A batched step whose tokens all belong to different sequences takes this part too (T > 1, no tickets): another
//    token's workgroup may read the row while it is written, but that cell is not visible to it - its score is replaced
//    by -inf and its V (old or new bytes, finite either way) is weighted by zero;
//  * merge: every workgroup publishes its chunk partial, then takes a ticket on a per-kv-head counter; the LAST arriver
//    merges the splits of its R heads exactly as flash_attn_combine_kernel does, writes the f32 rows and the quantised
//    activation of the attn_output mat-vec, and re-arms the counter.  Nobody waits: no spin, no co-residency needed.
struct DecodeFuse {
    const float *knew, *vnew;      // [G*D] un-rotated K and V of the token
    const int32_t *tok_cell;       // [1]
    unsigned *counters;            // [G] words ATT_SYNC_STRIDE apart (a 128-byte line each), zero between launches
    ActRows q;
    int want_q8k, want_q80;
    int neox;                      // rotary pairing (i, i + D / 2) instead of (2i, 2i + 1): qwen2-type files; the whole head rotates (n_rot == D)
    // diagnosis (MI355_ATTN_PROBE=1): 100 MHz wall-clock stamps.  [2 * wg], [2 * wg + 1] = start / partials-stored of every
    // workgroup (wg = sp * G + g); [4096 + 8 * g + k] = the merging workgroup of kv head g: ticket taken, weights done,
    // partials summed, outputs stored
    unsigned long long *probe;
};

// a wave quantises block gb of the token's attention output, its 256 values in LDS
template <bool COH>
__device__ __forceinline__ void decode_quant_block(const DecodeFuse &fz, const float *x, int gb, int lane) {
    const float4 v4 = *reinterpret_cast<const float4 *>(x + lane * 4);
    const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
    const int e0 = gb * 256 + lane * 4;
    if (fz.want_q8k) {
        uint32_t packed; int bs; float dq8;
        wave_quant_q8k(vv, lane, packed, bs, dq8);
        cst4<COH>(fz.q.qs + e0, packed);
        if ((lane & 3) == 0) cst2<COH>(fz.q.bsums + gb * 16 + (lane >> 2), (unsigned short)(int16_t)bs);
        if (lane == 0) cstf<COH>(fz.q.d + gb, dq8);
    }
    if (fz.want_q80) {
        uint32_t packed; float dd;
        wave_quant_q80(vv, packed, dd);
        cst4<COH>(fz.q.qs0 + e0, packed);
        if ((lane & 7) == 0) cst2<COH>(fz.q.d0 + gb * 8 + (lane >> 3), f2h(dd));
    }
}

// body of one (kv head g, chunk slot sp, token t) work item; 256 threads, every exit is workgroup-uniform
// COH (decode_mega.hip): q / K / V of the token come from other workgroups of the same launch and the results go to
// other workgroups of the same launch: those accesses are made device-coherent (dev_common.h) and the ticket is a relaxed
// atomic, instead of an agent-scope release / acquire whose cache-wide write-back and invalidate cost microseconds.
// D = 128 (default) or 64: head_dim; every lane role below is derived from it
// NS > 1: a workgroup of NS * 256 threads holds all chunks of R query heads from qh on, a chunk to 256 threads; their merge needs no ticket then (flash_attn_decode_whole_kernel)
template <int R, int TK, int TV, bool FUSED, bool COH = false, int D = 128, int NS = 1>
__device__ __forceinline__ void flash_attn_decode_item(const AttnArgs &a, const float *cs_table, int n_rot, const DecodeFuse &fz, int g, int sp, int t, int qh) {
    constexpr int C = 64, NB = D / 32;
    // (a q4_0 cache - TK = TV = T_Q4_0, head_dim 128 - keeps 16 nibble bytes per 32-block: a piece is a whole block, four lanes per cell)
    constexpr int KROW = TK == T_F16 ? 2 * D : TK == T_Q4_0 ? D / 2 : D, VROW = TV == T_Q4_0 ? D / 2 : D;   // bytes of a K row; bytes (halfs for f16) of a V row
    constexpr int LPC = KROW / 16;                           // lanes per cell in the score pass (16-byte pieces of a K row)
    constexpr int KP = C * LPC / 256;                       // 16-byte K pieces per thread
    constexpr int DQ = D / 4, NCG = 256 / DQ, CPG = C / NCG;   // P.V pass: DQ lanes of 4 dims, NCG cell groups of CPG cells
    __shared__ __attribute__((aligned(16))) float qf_[NS][R * D];         // rotated q (f16-rounded for an f16 cache)
    __shared__ __attribute__((aligned(16))) int8_t qc_[NS][R * D];        // q8_0 codes of q
    __shared__ float qd_[NS][R * NB];
    __shared__ __attribute__((aligned(16))) float S_[NS][R * C];          // [cell][head]: a cell's weights are read together
    // (the f16 scores and P V multiply and add in one instruction: with [head][cell] and two of them ticks of 4, 16 and 32 conversations, 32 / 8 heads of 128, took 7.40, 14.2 and 23.1 us a layer
    // instead of 7.17, 13.8 and 21.5, sixteen with 32 / 4 heads of 64 18.1 instead of 16.9 to 17.5: the chunk's arithmetic is a chain of one workgroup)
    __shared__ float ml_[NS][R * 2];
    __shared__ int vis_[NS][C];
    __shared__ uint32_t ksc_[NS][C * NB / 2], vsc_[NS][C * NB / 2];           // f16 block scales of the chunk
    __shared__ __attribute__((aligned(16))) float accs_[NS][NCG * R * D];
    __shared__ __attribute__((aligned(16))) uint8_t newk_[NS][D * 2], newv_[NS][D * 2];   // the token's own cache row (codes or f16)
    __shared__ uint32_t newkd_[NS][2], newvd_[NS][2];                                      // its f16 block scales, two per word
    __shared__ int last_flag, any_[NS];
    const int sub = NS > 1 ? __builtin_amdgcn_readfirstlane(tid_now() >> 8) : 0, tid = NS > 1 ? tid_now() & 255 : tid_now(), lane = tid & 63, wave = tid >> 6;
    float *const qf = qf_[sub], *const qd = qd_[sub], *const S = S_[sub], *const ml = ml_[sub], *const accs = accs_[sub];
    int8_t *const qc = qc_[sub];
    int *const vis = vis_[sub];
    uint32_t *const ksc = ksc_[sub], *const vsc = vsc_[sub], *const newkd = newkd_[sub], *const newvd = newvd_[sub];
    uint8_t *const newk = newk_[sub], *const newv = newv_[sub];
    const int n_ctx = a.n_ctx, H = a.H;
    if (FUSED && fz.probe && tid == 0) fz.probe[2 * (sp * a.G + g)] = wall_clock64();
    int chunk = sp;
    bool live = true;
    if (a.tok_chunks) {                                        // walk this token's chunk list only (sequences own cache regions)
        live = sp < a.tok_nchunks[t];
        if (NS == 1 && !live) return;
        if (live) chunk = a.tok_chunks[(size_t)t * a.chunk_stride + sp];
    } else if (NS > 1) live = sp < a.splits;
    if (!live) chunk = 0;                                      // (addresses that exist; nothing of it is visible)
    const int c_lo = chunk * C;
    const size_t head_row0 = (size_t)g * n_ctx;

    // ---- issue every global load of the workgroup
    int cpos = -1;
    unsigned long long cseq = 0;
    if (tid < C && c_lo + tid < n_ctx) { cpos = a.cell_pos[c_lo + tid]; cseq = a.cell_seq[c_lo + tid]; }
    const int32_t tpos = a.tok_pos[t];
    const int tseq = a.tok_seq[t];
    if (a.T > 1 && !a.tok_chunks) {
        // batched steps (one token per sequence) without chunk lists: most chunks hold other sequences' cells only.  Decide that before
        // touching K / V: such a chunk publishes (m, l) = (-inf, 0) and leaves; the merge skips it.  (A list names the chunks that hold cells of the token's sequence, and
        // the cells' answer would be a trip to memory in front of K's and V's)
        const int mine = (tid < C && cpos >= 0 && cpos <= tpos && ((cseq >> tseq) & 1ull)) ? 1 : 0;
        if (!__syncthreads_or(mine)) {
            if (tid < R) {
                float *dst = a.part + (((size_t)t * H + (size_t)qh + tid) * a.splits + sp) * att_rec(D);
                dst[D] = -INFINITY; dst[D + 1] = 0.0f;
            }
            return;
        }
    }
    // q pairs: R * D / 2 pairs, pair pp -> (head r = pp / (D / 2), i = pp % (D / 2)); NORM pairing (2i, 2i+1)
    constexpr int HP = D / 2, NPAIR = R * HP, PPT = (NPAIR + 255) / 256;
    float2 qv[PPT], csv[PPT];
#pragma unroll
    for (int j = 0; j < PPT; j++) {
        const int pp = tid + 256 * j;
        if (pp < NPAIR) {
            const int r = pp / HP, i = pp % HP;
            if (fz.neox) {                                      // the pair's halves lie D / 2 apart
                const int o = (int)((((size_t)t * H + (size_t)qh + r) * D + i) * 4);
                qv[j] = make_float2(__uint_as_float(cld4<COH>(a.q, o)), __uint_as_float(cld4<COH>(a.q, o + HP * 4)));
            } else {
                const coh_u32x2 qq = cld8<COH>(a.q, (int)((((size_t)t * H + (size_t)qh + r) * D + 2 * i) * 4));
                qv[j] = make_float2(__uint_as_float(qq.x), __uint_as_float(qq.y));
            }
            csv[j] = (2 * i < n_rot) ? *reinterpret_cast<const float2 *>(cs_table + (size_t)t * n_rot + 2 * i) : make_float2(1.0f, 0.0f);
        }
    }
    uint4 kreg[KP];
#pragma unroll
    for (int j = 0; j < KP; j++) {
        const int p = tid + 256 * j;
        int cell = c_lo + p / LPC;
        if (cell >= n_ctx) cell = n_ctx - 1;
        const size_t rowi = head_row0 + cell;
        if (TK == T_F16) kreg[j] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(a.kv.k) + rowi * D + (p % LPC) * 8);
        else kreg[j] = *reinterpret_cast<const uint4 *>(a.kv.k + rowi * KROW + (p % LPC) * 16);
    }
    const int dq = tid % DQ, cg = tid / DQ;
    uint2 vreg[CPG];
#pragma unroll
    for (int i = 0; i < CPG; i++) {
        int cell = c_lo + cg + NCG * i;
        if (cell >= n_ctx) cell = n_ctx - 1;
        const size_t rowi = head_row0 + cell;
        if (TV == T_F16) vreg[i] = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(a.kv.v) + rowi * D + dq * 4);
        else if (TV == T_Q4_0) {            // dims 4 dq .. + 3 of block dq >> 3: the low or the high nibbles of four consecutive bytes, kept one per byte
            const int e0 = (dq * 4) & 31;
            const uint32_t w = *reinterpret_cast<const uint32_t *>(a.kv.v + rowi * VROW + (dq >> 3) * 16 + (e0 & 15));
            vreg[i].x = (e0 < 16 ? w : (w >> 4)) & 0x0f0f0f0fu; vreg[i].y = 0;
        }
        else { vreg[i].x = *reinterpret_cast<const uint32_t *>(a.kv.v + rowi * D + dq * 4); vreg[i].y = 0; }
    }
    uint32_t ks2 = 0, vs2 = 0;
    if (tid < C * NB / 2) {                                            // NB / 2 words (two f16 scales each) per cell
        int cell = c_lo + tid / (NB / 2);
        if (cell >= n_ctx) cell = n_ctx - 1;
        if (TK != T_F16) ks2 = *reinterpret_cast<const uint32_t *>(a.kv.kd + (head_row0 + cell) * NB + (tid % (NB / 2)) * 2);
        if (TV != T_F16) vs2 = *reinterpret_cast<const uint32_t *>(a.kv.vd + (head_row0 + cell) * NB + (tid % (NB / 2)) * 2);
    }

    // ---- FUSED: this token's K/V row (wave 0: lanes 0..31 rotate + convert K, lanes 32..63 convert V; 4 elements each)
    int own_cl = -1;                                   // chunk-local index of the token's cell, if this chunk holds it
    if (FUSED) {
        const int cellnew = fz.tok_cell[t];                      // (t = 0 in a single-token step)
        if (live && cellnew >= c_lo && cellnew < c_lo + C) own_cl = cellnew - c_lo;
        if (own_cl >= 0 && wave == 0 && (lane & 31) < DQ) {      // lanes 0 .. DQ - 1: K, lanes 32 .. 32 + DQ - 1: V (whole 8-lane groups either way)
            const bool isk = lane < 32;
            const int dd = (lane & 31) * 4;
            float4 x4;
            {
                const coh_u32x4 xx = cld16<COH>(isk ? fz.knew : fz.vnew, ((t * a.G + g) * D + dd) * 4);
                x4 = make_float4(__uint_as_float(xx.x), __uint_as_float(xx.y), __uint_as_float(xx.z), __uint_as_float(xx.w));
            }
            if (fz.neox) {
                // NEOX pairing: element e < D / 2 rotates with e + D / 2, which sits DQ / 2 lanes further on (both K lanes and V lanes run the exchange)
                const float p0 = __shfl_xor(x4.x, DQ / 2), p1 = __shfl_xor(x4.y, DQ / 2), p2 = __shfl_xor(x4.z, DQ / 2), p3 = __shfl_xor(x4.w, DQ / 2);
                if (isk) {
                    const bool lo = dd < HP;
                    const float *cp = cs_table + (size_t)t * n_rot + 2 * (lo ? dd : dd - HP);              // (c, s) of pairs dd' .. dd' + 3
                    const float4 ca = *reinterpret_cast<const float4 *>(cp), cb = *reinterpret_cast<const float4 *>(cp + 4);
                    if (lo) { x4.x = x4.x * ca.x - p0 * ca.y; x4.y = x4.y * ca.z - p1 * ca.w; x4.z = x4.z * cb.x - p2 * cb.y; x4.w = x4.w * cb.z - p3 * cb.w; }
                    else { x4.x = p0 * ca.y + x4.x * ca.x; x4.y = p1 * ca.w + x4.y * ca.z; x4.z = p2 * cb.y + x4.z * cb.x; x4.w = p3 * cb.w + x4.w * cb.z; }
                }
            } else if (isk && dd < n_rot) {
                const float4 cs = *reinterpret_cast<const float4 *>(cs_table + (size_t)t * n_rot + dd);   // c0 s0 c1 s1
                const float x0 = x4.x, x1 = x4.y, x2 = x4.z, x3 = x4.w;
                x4.x = x0 * cs.x - x1 * cs.y; x4.y = x0 * cs.y + x1 * cs.x;
                x4.z = x2 * cs.z - x3 * cs.w; x4.w = x2 * cs.w + x3 * cs.z;
            }
            const float xa[4] = {x4.x, x4.y, x4.z, x4.w};
            const size_t rowi = head_row0 + cellnew;
            const int TT = isk ? TK : TV;              // (TK, TV are compile-time; the select folds per branch below)
            uint32_t packed = 0; float dsc = 0.0f;
            if (TK == T_Q4_0) wave_quant_q40(xa, lane, packed, dsc);            // (TK = TV = T_Q4_0 only)
            else if (TK != T_F16 || TV != T_F16) wave_quant_q80(xa, packed, dsc);   // whole wave takes part (8-lane groups)
            if (TT == T_Q4_0) {
                const uint32_t hi = __shfl_xor(packed, 4, 64);                  // the lane four further on holds elements j + 16 of the block
                if ((lane & 4) == 0) {
                    const uint32_t bytes = packed | (hi << 4);
                    const int off = (dd >> 5) * 16 + (dd & 15);
                    *reinterpret_cast<uint32_t *>((isk ? newk : newv) + off) = bytes;
                    *reinterpret_cast<uint32_t *>((isk ? a.kv.k : a.kv.v) + rowi * (D / 2) + off) = bytes;
                }
                if ((lane & 7) == 0) {
                    const uint16_t hd = f2h(dsc);
                    (isk ? a.kv.kd : a.kv.vd)[rowi * NB + (dd >> 5)] = hd;
                    reinterpret_cast<uint16_t *>(isk ? newkd : newvd)[dd >> 5] = hd;
                }
            } else if (TT == T_F16) {
                uint2 o; o.x = (uint32_t)f2h(xa[0]) | ((uint32_t)f2h(xa[1]) << 16); o.y = (uint32_t)f2h(xa[2]) | ((uint32_t)f2h(xa[3]) << 16);
                *reinterpret_cast<uint2 *>((isk ? newk : newv) + dd * 2) = o;
                *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(isk ? a.kv.k : a.kv.v) + rowi * D + dd) = o;
            } else {
                *reinterpret_cast<uint32_t *>((isk ? newk : newv) + dd) = packed;
                *reinterpret_cast<uint32_t *>((isk ? a.kv.k : a.kv.v) + rowi * D + dd) = packed;
                if ((lane & 7) == 0) {
                    const uint16_t hd = f2h(dsc);
                    (isk ? a.kv.kd : a.kv.vd)[rowi * NB + (dd >> 5)] = hd;
                    reinterpret_cast<uint16_t *>(isk ? newkd : newvd)[dd >> 5] = hd;
                }
            }
        }
    }

    // ---- q: rotate, convert
    if (tid < C) {
        const bool v = live && cpos >= 0 && cpos <= tpos && ((cseq >> tseq) & 1ull);
        vis[tid] = v ? 1 : 0;
        if (NS > 1) { const bool some = __ballot(v) != 0; if (tid == 0) any_[sub] = some; }
    }
    if (tid < C * NB / 2) { ksc[tid] = ks2; vsc[tid] = vs2; }
#pragma unroll
    for (int j = 0; j < PPT; j++) {
        const int pp = tid + 256 * j;
        if (pp < NPAIR) {
            const float x0 = qv[j].x, x1 = qv[j].y, c = csv[j].x, s = csv[j].y;
            float y0 = x0 * c - x1 * s, y1 = x0 * s + x1 * c;
            if (TK == T_F16) { y0 = h2f(f2h(y0)); y1 = h2f(f2h(y1)); }
            if (fz.neox) { const int r = pp / HP, i = pp % HP; qf[r * D + i] = y0; qf[r * D + i + HP] = y1; }
            else *reinterpret_cast<float2 *>(qf + 2 * pp) = make_float2(y0, y1);
        }
    }
    __syncthreads();
    if (FUSED && own_cl >= 0) {   // workgroup-uniform: use the row just produced instead of what the cache held before
        if (tid < NB / 2) {
            if (TK != T_F16) ksc[own_cl * (NB / 2) + tid] = newkd[tid];
            if (TV != T_F16) vsc[own_cl * (NB / 2) + tid] = newvd[tid];
        }
#pragma unroll
        for (int j = 0; j < KP; j++) {
            const int p = tid + 256 * j;
            if (p / LPC == own_cl) kreg[j] = *reinterpret_cast<const uint4 *>(newk + (p % LPC) * 16);
        }
#pragma unroll
        for (int i = 0; i < CPG; i++) {
            if (cg + NCG * i == own_cl) {
                if (TV == T_F16) vreg[i] = *reinterpret_cast<const uint2 *>(newv + dq * 8);
                else if (TV == T_Q4_0) {
                    const int e0 = (dq * 4) & 31;
                    const uint32_t w = *reinterpret_cast<const uint32_t *>(newv + (dq >> 3) * 16 + (e0 & 15));
                    vreg[i].x = (e0 < 16 ? w : (w >> 4)) & 0x0f0f0f0fu; vreg[i].y = 0;
                }
                else { vreg[i].x = *reinterpret_cast<const uint32_t *>(newv + dq * 4); vreg[i].y = 0; }
            }
        }
    }
    if (TK != T_F16) {   // q8_0 of the rotated q: 4 values per thread, 8-lane groups
        for (int e0 = tid * 4; e0 < R * D; e0 += 1024) {
            const float4 v4 = *reinterpret_cast<const float4 *>(qf + e0);
            const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
            uint32_t packed; float d;
            wave_quant_q80(vv, packed, d);
            *reinterpret_cast<uint32_t *>(qc + e0) = packed;
            if ((lane & 7) == 0) qd[e0 >> 5] = h2f(f2h(d));
        }
        __syncthreads();
    }

    // ---- scores
    const bool any = NS == 1 || __builtin_amdgcn_readfirstlane(any_[sub]) != 0;          // (a chunk without a visible cell: weights of zero, none of the arithmetic)
#pragma unroll
    for (int j = 0; j < KP; j++) {
        if (!any) break;
        const int p = tid + 256 * j;
        const int cl = p / LPC, piece = p % LPC;
        float sc[R];
        if (TK == T_F16) {
            const uint32_t kw[4] = {kreg[j].x, kreg[j].y, kreg[j].z, kreg[j].w};
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float *qq = qf + r * D + piece * 8;
                float s = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s = __builtin_fmaf(h2f((uint16_t)(kw[i] & 0xffff)), qq[2 * i], s);
                    s = __builtin_fmaf(h2f((uint16_t)(kw[i] >> 16)), qq[2 * i + 1], s);
                }
                s += dpp_f<DPP_QP_1032>(s); s += dpp_f<DPP_QP_2301>(s); s += dpp_f<DPP_HALF_MIRROR>(s);      // 8 lanes
                if (LPC == 16) s += dpp_f<DPP_MIRROR>(s);
                sc[r] = s;
            }
        } else if (TK == T_Q4_0) {   // vec_dot_q4_0_q8_0: piece = 32-block; codes nibble - 8 against the q8_0 codes of q, low nibbles = elements 0 .. 15
            const uint32_t kpair = ksc[cl * (NB / 2) + (piece >> 1)];
            const float dk = h2f((uint16_t)((piece & 1) ? (kpair >> 16) : (kpair & 0xffff)));
            const uint32_t kw[4] = {kreg[j].x, kreg[j].y, kreg[j].z, kreg[j].w};
            uint32_t klo[4], khi[4];
#pragma unroll
            for (int w = 0; w < 4; w++) { klo[w] = nib_to_i8x4(kw[w] & 0x0f0f0f0fu); khi[w] = nib_to_i8x4((kw[w] >> 4) & 0x0f0f0f0fu); }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint4 q0 = *reinterpret_cast<const uint4 *>(qc + r * D + piece * 32), q1 = *reinterpret_cast<const uint4 *>(qc + r * D + piece * 32 + 16);
                int s = 0;
                s = dot4(klo[0], q0.x, s); s = dot4(klo[1], q0.y, s); s = dot4(klo[2], q0.z, s); s = dot4(klo[3], q0.w, s);
                s = dot4(khi[0], q1.x, s); s = dot4(khi[1], q1.y, s); s = dot4(khi[2], q1.z, s); s = dot4(khi[3], q1.w, s);
                float f = (float)s * (dk * qd[r * NB + piece]);
                f += dpp_f<DPP_QP_1032>(f); f += dpp_f<DPP_QP_2301>(f);                                 // the cell's four blocks
                sc[r] = f;
            }
        } else {
            const uint32_t kpair = ksc[cl * (NB / 2) + (piece >> 2)];
            const float dk = h2f((uint16_t)(((piece >> 1) & 1) ? (kpair >> 16) : (kpair & 0xffff)));
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint4 qq = *reinterpret_cast<const uint4 *>(qc + r * D + piece * 16);
                int s = 0;
                s = dot4(kreg[j].x, qq.x, s); s = dot4(kreg[j].y, qq.y, s); s = dot4(kreg[j].z, qq.z, s); s = dot4(kreg[j].w, qq.w, s);
                s += dpp_i<DPP_QP_1032>(s);                    // both halves of the 32-block (integer)
                float f = (piece & 1) ? 0.0f : (float)s * (dk * qd[r * NB + (piece >> 1)]);
                f += dpp_f<DPP_QP_1032>(f); f += dpp_f<DPP_QP_2301>(f);                                 // 4 lanes
                if (LPC == 8) f += dpp_f<DPP_HALF_MIRROR>(f);                                            // 8 lanes
                sc[r] = f;
            }
        }
        if (piece == 0) {
            const bool v = vis[cl] != 0;
#pragma unroll
            for (int r = 0; r < R; r++) S[cl * R + r] = v ? sc[r] * a.scale : -INFINITY;
        }
    }
    __syncthreads();

    // ---- softmax of the chunk: wave w -> heads w, w+4, ...; lane = cell
    for (int r = wave; r < R; r += 4) {
        const float s = any ? S[lane * R + r] : -INFINITY;
        const float m = wave_max(s);
        const float p = (s == -INFINITY) ? 0.0f : expf(s - m);
        const float l = wave_sum(p);
        S[lane * R + r] = p;
        if (lane == 0) { ml[2 * r] = m; ml[2 * r + 1] = l; }
    }
    __syncthreads();

    // ---- P.V
    float acc[R][4];
#pragma unroll
    for (int r = 0; r < R; r++) { acc[r][0] = acc[r][1] = acc[r][2] = acc[r][3] = 0.0f; }
#pragma unroll
    for (int i = 0; i < CPG; i++) {
        if (!any) break;
        const int cl = cg + NCG * i;
        float v4[4];
        if (TV == T_F16) {
            v4[0] = h2f((uint16_t)(vreg[i].x & 0xffff)); v4[1] = h2f((uint16_t)(vreg[i].x >> 16));
            v4[2] = h2f((uint16_t)(vreg[i].y & 0xffff)); v4[3] = h2f((uint16_t)(vreg[i].y >> 16));
        } else {
            const uint32_t vpair = vsc[cl * (NB / 2) + (dq >> 4)];
            const float dv = h2f((uint16_t)(((dq >> 3) & 1) ? (vpair >> 16) : (vpair & 0xffff)));
            const uint32_t w = TV == T_Q4_0 ? nib_to_i8x4(vreg[i].x) : vreg[i].x;
            v4[0] = (float)(int8_t)(w & 0xff) * dv; v4[1] = (float)(int8_t)((w >> 8) & 0xff) * dv;
            v4[2] = (float)(int8_t)((w >> 16) & 0xff) * dv; v4[3] = (float)(int8_t)(w >> 24) * dv;
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float p = S[cl * R + r];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[r][e] = __builtin_fmaf(v4[e], p, acc[r][e]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        *reinterpret_cast<float4 *>(accs + ((size_t)cg * R + r) * D + dq * 4) = make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
    __syncthreads();
    for (int e = tid; e < R * D; e += 256) {
        const int r = e / D, d = e - r * D;
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < NCG; j++) s += accs[((size_t)j * R + r) * D + d];
        if (NS > 1) { S[e] = s; continue; }                   // (the chunk's weights are spent)
        float *dst = a.part + (((size_t)t * H + (size_t)qh + r) * a.splits + sp) * att_rec(D);
        cstf<COH>(dst + d, s);
        if (d == 0) { cstf<COH>(dst + D, ml[2 * r]); cstf<COH>(dst + D + 1, ml[2 * r + 1]); }
    }
    if (!FUSED) return;
    if constexpr (NS > 1) {
        // every chunk is here: the merge below, of records in LDS
        static_assert(COH == false && D <= C && (R * D) % 256 == 0 && R <= 4 * NS && R * D <= 256 * NS, "a wave to a head, a thread to an output, whole blocks");
        if (fz.probe && tid == 0) fz.probe[2 * (sp * a.G + g) + 1] = wall_clock64();
        __syncthreads();
        const int all = tid_now(), wv = __builtin_amdgcn_readfirstlane(all >> 6);
        if (fz.probe && all == 0) fz.probe[4096 + 8 * g] = wall_clock64();
        float *const wgt = accs_[0], *const merged = qf_[0];
        if (wv < R) {
            const float m = lane < NS ? ml_[lane < NS ? lane : 0][2 * wv] : -INFINITY, l = lane < NS ? ml_[lane < NS ? lane : 0][2 * wv + 1] : 0.0f;
            const float M = wave_max(m);
            const float w = m != -INFINITY ? expf(m - M) : 0.0f;
            const float den = wave_sum(w * l);
            if (lane < NS) wgt[wv * 64 + lane] = w * (1.0f / den);
        }
        __syncthreads();
        if (fz.probe && all == 0) fz.probe[4096 + 8 * g + 1] = wall_clock64();
        if (all < R * D) {
            const int r = all / D;
            float s = 0.0f;
#pragma unroll
            for (int c = 0; c < NS; c++) s += wgt[r * 64 + c] * S_[c][all];
            merged[all] = s;
            a.out[(size_t)qh * D + all] = s;
        }
        __syncthreads();
        if (fz.probe && all == 0) fz.probe[4096 + 8 * g + 2] = wall_clock64();
        if (wv < (R * D) >> 8 && (fz.want_q8k || fz.want_q80)) decode_quant_block<COH>(fz, merged + wv * 256, ((qh * D) >> 8) + wv, lane);
        if (fz.probe && wv == 0) {                            // (the block's wave)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (lane == 0) fz.probe[4096 + 8 * g + 3] = wall_clock64();
        }
        return;
    }
    if (fz.counters == nullptr) return;               // store-fused only: the merge runs as its own launch (batched steps: in this launch it takes as long, ticks of 2 to 16 tokens 1 % slower to 1 % faster)
    if (fz.probe && tid == 0) fz.probe[2 * (sp * a.G + g) + 1] = wall_clock64();

    // ---- FUSED: ticket; the last workgroup of this kv head merges.  The merge also quantises whole 256-element blocks of
    // the attention output, so with one 128-wide query head per kv head (R = 1, multi-head attention) TWO neighbouring kv
    // heads share a ticket and the last arriver of the pair merges both: GP kv heads per ticket, RM = GP * R heads merged.
    // (in general the smallest number of kv heads whose R * D outputs fill whole blocks: 256 / gcd(R * D, 256) - two for 3, 5 or 7 query heads of 128 per kv head)
    constexpr int GP = 256 / ((R * D) % 256 == 0 ? 256 : (R * D) % 128 == 0 ? 128 : (R * D) % 64 == 0 ? 64 : 32);
    constexpr int RM = R * GP;
    const int gq = g / GP;                                     // ticket group
    const int hb = gq * RM;                                    // its first query head
    const int stride_s = a.splits;                             // workspace stride; with a chunk list fewer slots are in use
    const int splits = a.tok_nchunks ? a.tok_nchunks[0] : a.splits;
    // every wave's partial stores must have reached L2 before thread 0 releases them device-wide: __syncthreads() fences
    // LDS only (hipcc emitted no vmcnt wait before the barrier here), so each wave drains its own stores first
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (a workgroup-scope release fence compiles to nothing on this target)
    __syncthreads();
    if (tid == 0) {
        // ONE release per workgroup (the barrier ordered the other waves' stores before it), then the ticket
        const unsigned old = COH ? __hip_atomic_fetch_add(fz.counters + gq * ATT_SYNC_STRIDE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                 : __hip_atomic_fetch_add(fz.counters + gq * ATT_SYNC_STRIDE, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        last_flag = (old == (unsigned)(splits * GP) - 1u) ? 1 : 0;
        if (last_flag) __hip_atomic_store(fz.counters + gq * ATT_SYNC_STRIDE, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-arm
    }
    __syncthreads();
    if (!last_flag) return;
    if (fz.probe && tid == 0) fz.probe[4096 + 8 * g] = wall_clock64();
    float *merged = accs;                              // [RM * D]
    float *wgt = GP > 1 ? accs + RM * D : S;           // [RM][64] split weights (S is free now, but holds R * C floats only)
    // The merge is a chain of memory round trips (~1.5 us each: the partials come from other XCDs).  Every output still
    // sums its splits in order (the combine kernel's arithmetic), but the partials of the first UB splits of all of this
    // thread's outputs are requested BEFORE the (m, l) pairs, so the weight computation runs under them: ticket, one trip
    // for (m, l) + UB splits, one more per further UB (it was ticket + (m, l) + one trip per 8 splits and output).  UB by the splits there are: a load past them is one more
    // trip of the fabric's (us a launch of a step, 4 kv heads of 8 heads of 64 behind 93 cells: 10.0 with thirty-two loads an output for four splits and the argument
    // segment read field by field, 8.6 in a replayed step; launched eagerly 9.5)
    constexpr int NE = (RM * D + 255) / 256;
    float macc[NE];
    const float *pp[NE];
    int wr[NE];
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = tid + 256 * j < RM * D ? tid + 256 * j : 0, r = e / D, d = e - r * D;
        pp[j] = a.part + ((size_t)hb + r) * stride_s * att_rec(D) + d;
        wr[j] = r * 64;
        macc[j] = 0.0f;
    }
    const auto merge = [&](auto ub) __attribute__((always_inline)) {
        constexpr int UB = decltype(ub)::value;        // (NE * UB partials in registers per thread)
        float x[NE][UB];
        auto request = [&](int s0) {
#pragma unroll
            for (int u = 0; u < UB; u++) {
                const int s2 = s0 + u < splits ? s0 + u : splits - 1;          // clamped: straight-line loads
#pragma unroll
                for (int j = 0; j < NE; j++) x[j][u] = __hip_atomic_load(pp[j] + (size_t)s2 * att_rec(D), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        request(0);
        for (int r = wave; r < RM; r += 4) {           // same arithmetic as flash_attn_combine_kernel
            const float *p = a.part + ((size_t)hb + r) * stride_s * att_rec(D);
            float m = -INFINITY, l = 0.0f;
            if (lane < splits) {
                m = __hip_atomic_load(p + (size_t)lane * att_rec(D) + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                l = __hip_atomic_load(p + (size_t)lane * att_rec(D) + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            const float M = wave_max(m);
            const float w = (lane < splits && m != -INFINITY) ? expf(m - M) : 0.0f;
            const float den = wave_sum(w * l);
            const float inv = 1.0f / den;
            wgt[r * 64 + lane] = w * inv;
        }
        __syncthreads();
        if (fz.probe && tid == 0) fz.probe[4096 + 8 * g + 1] = wall_clock64();
        for (int s0 = 0;;) {
#pragma unroll
            for (int u = 0; u < UB; u++) {
                if (s0 + u < splits) {                                         // workgroup-uniform
#pragma unroll
                    for (int j = 0; j < NE; j++) macc[j] += wgt[wr[j] + s0 + u] * x[j][u];
                }
            }
            s0 += UB;
            if (s0 >= splits) break;
            request(s0);
        }
    };
    if (splits <= 4) merge(std::integral_constant<int, 4>());
    else if (splits <= 12) merge(std::integral_constant<int, 12>());
    else merge(std::integral_constant<int, (NE > 4 ? 16 : 32)>());
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = tid + 256 * j;
        if (e < RM * D) { merged[e] = macc[j]; a.out[(size_t)hb * D + e] = macc[j]; }
    }
    if (fz.probe && tid == 0) fz.probe[4096 + 8 * g + 2] = wall_clock64();
    __syncthreads();
    constexpr int NBLK = (RM * D) >> 8;                // 256-blocks this ticket group owns in the H*D row
    if (wave < NBLK && (fz.want_q8k || fz.want_q80)) {
        for (int b = wave; b < NBLK; b += 4) {
            decode_quant_block<COH>(fz, merged + b * 256, ((hb * D) >> 8) + b, lane);
        }
    }
    if (fz.probe) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (tid == 0) fz.probe[4096 + 8 * g + 3] = wall_clock64();
    }
}

// (the argument segment is cold at every launch: a read of each of its lines at once, instead of one behind the other where a field is first used)
__device__ __forceinline__ void decode_args_at_once() {
    struct KArgs { AttnArgs a; const float *cs; int n_rot; DecodeFuse fz; };
    const __attribute__((address_space(4))) unsigned *ka = (const __attribute__((address_space(4))) unsigned *)__builtin_amdgcn_kernarg_segment_ptr();
    unsigned acc = 0;
#pragma unroll
    for (int i = 0; i < (int)((sizeof(KArgs) + 63) / 64); i++) acc ^= ka[i * 16];
    asm volatile("" :: "s"(acc));
}

template <int R, int TK, int TV, bool FUSED, bool COH = false, int D = 128>
__global__ __launch_bounds__(256) void flash_attn_decode_kernel(const AttnArgs a, const float *cs_table, int n_rot, const DecodeFuse fz) {
    decode_args_at_once();
    flash_attn_decode_item<R, TK, TV, FUSED, COH, D>(a, cs_table, n_rot, fz, blockIdx.x, blockIdx.y, blockIdx.z, blockIdx.x * R);
}

// A single token's step over few cells: a workgroup holds R of a kv head's query heads (of H / G: the others' workgroups read the same chunks) and all WHOLE_NS chunks, so that a record, the
// ticket and the other workgroups' records (a trip of the fabric each) leave the chain.  The same arithmetic in the same order.  Four heads of 64: their results are one block of 256 values to
// quantise, and four chunks of them are a CU's threads.  us a launch, 32 / 4 heads of 64, f16 cache, behind 20, 93 and 250 cells: 6.3, 6.7 and 7.1; with a workgroup a chunk and the ticket 8.7
// (six layers' step 220 -> 203, 206 and 212)
constexpr int WHOLE_NS = 4, WHOLE_R = 4, WHOLE_D = 64;
template <int TK, int TV, bool PROBE>
__global__ __launch_bounds__(256 * WHOLE_NS) void flash_attn_decode_whole_kernel(const AttnArgs a, const float *cs_table, int n_rot, const DecodeFuse fz_) {
    decode_args_at_once();
    DecodeFuse fz = fz_;
    if (!PROBE) fz.probe = nullptr;                            // (looked at behind every phase it is 0.1 us of the 7.1 behind 250 cells)
    const int parts = a.H / a.G / WHOLE_R;
    flash_attn_decode_item<WHOLE_R, TK, TV, true, false, WHOLE_D, WHOLE_NS>(a, cs_table, n_rot, fz, blockIdx.x / parts, __builtin_amdgcn_readfirstlane(tid_now() >> 8), 0, blockIdx.x * WHOLE_R);
}

}  // namespace mi355
