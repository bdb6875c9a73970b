// Gated GQA decode attention over a bf16 KV cache, split over 256-slot chunks.
//
// Math (speccheck/specimpl.py:320-397): de-interleave [q | gate] per head; zero-centred
// RMSNorm on q and k per head; rope on dims 0..63 (pairs i, i+32, theta 1e7) in f32;
// append k (post-rope) and v at the row's cache slot; scores q.K / 16 in f32; softmax in
// f32; weights rounded to bf16; P.V with f32 accumulation rounded to bf16; times
// bf16(sigmoid(gate)). GQA: query head i reads kv head i / 4.
// Replaces engine/kernels_attn.cpp:415-1108 (prep, core, combine) of the reference.
//
// Four launches per layer (batched lanes with short enough contexts: prep + one fused
// kernel, attn_fused):
//   attn_prep   (row, head)         q norm+rope -> f32 scratch; k norm+rope, v -> cache
//   attn_scores (row, kv head, chunk) scores on MFMA -> scratch, per-chunk (max, sum e^(s-max))
//   attn_pv     (row, kv head, 128-slot part) global (max, sum) from the chunk stats,
//               p = bf16(e/l), partial P.V per part on MFMA (V cache in 8-slot groups)
//   attn_combine (row, q head)      sum of the parts in order, bf16, times bf16(sigmoid(gate))
// plus attn_rows and attn_seg_* (MTP verify: a lane's rows in one block, or in one block per segment)
// and attn_prompt (prompt waves).
// The k cache holds bf16(k post-rope); the reference's torch path keeps it in f32, so
// k's rotated dims carry one extra bf16 rounding here (the cache layout is bf16 by design).
#include <algorithm>
#include <type_traits>

#include "q35_common.h"
#include "q35_kernels.h"

namespace q35 {

constexpr int kChunk = 256;
// attn_rows<T, W>: the top parts (128 slots) whose scores fit the block's dynamic LDS beside
// the slice stats keep them there -- W = 4: two blocks per CU (80 KiB each, less the static q
// staging and ml), at most 8 parts; W = 8: one block per CU, at most 24 parts
constexpr int kRowsLdsDyn4 = 80 * 1024 - 16480, kRowsLdsDyn8 = 160 * 1024 - 16480;
__host__ __device__ constexpr int rows_lds_parts(int T, int max_chunks, int W) {
    return max(0, min(W == 8 ? 24 : 8, ((W == 8 ? kRowsLdsDyn8 : kRowsLdsDyn4) - T * 4 * 8 * max_chunks * 4) /
                                           (T * 4 * 128 * 4)));
}
__host__ __device__ constexpr size_t rows_lds_bytes(int T, int max_chunks, int W) {
    return (size_t)T * 4 * (8 * max_chunks + 128 * rows_lds_parts(T, max_chunks, W)) * 4;
}
// attn_fused<*, 2>: dynamic LDS of its two items, the CU's 160 KiB less both halves' static
// arrays (ubuf, ml, nparts)
constexpr int kFused2MaxLds = 160 * 1024 - 16464;

// Scores on MFMA: a wave takes 16 cache slots per v_mfma_f32_16x16x32_bf16 chain with the
// K rows as the A operand (step s of lane (slot t, group g) carries dims s*32 + g*8 .. +8;
// the K cache is stored in exactly that order, q35_common.h kv_tiled_offset, so each load
// instruction reads one contiguous KiB) and B = [q_hi(4 heads) |
// q_lo(4 heads) | 0], q_hi = bf16(q), q_lo = bf16(q - q_hi), so s = C[t][h] + C[t][h+4]
// carries q to ~2^-16 relative. A chunk = 4 waves x 64 slots.
//
// The chunk score pass, the part P.V pass and the part sum are device functions shared by
// the split kernels (any batch, any context) and the fused per-lane kernel (batched lanes,
// contexts that fit LDS), so both give the same bits.

// q fragments of kv group j for row r (all 256 threads; contains a barrier).
__device__ __forceinline__ void load_q_frags(const AttnArgs& a, int r, int j, uint16_t (*qb)[256],
                                             q35_u32x4* qf) {
    const int tid = threadIdx.x & 255, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const float* q = a.q + ((size_t)r * kNq + 4 * j) * 256;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const float qv = q[h * 256 + tid];
        const uint16_t hi = f2bf(qv);
        qb[h][tid] = hi;
        qb[4 + h][tid] = f2bf(qv - bf2f(hi));
        qb[8 + h][tid] = 0;
        qb[12 + h][tid] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const q35_u32x4*)&qb[n][s * 32 + g * 8];
}

// Scores of chunk c (slots c*256 .. +256, masked beyond `slot`) -> dst[h * dst_stride + t],
// chunk stats (max, sum e^(s - max)) -> stats[h * stats_stride + 2c .. +1]. Contains barriers.
// K fragments of sub-tile st of 64-slot slice q for this lane: K tile 4q + st of the tiled
// cache, step s = one contiguous KiB (the tile index is clamped to `slot`'s tile; slots past
// `slot` are masked later).
// NT: nontemporal loads (streamed once: one row per lane); cached when the lane's several rows
// (MTP verify rows) read the same K/V from L2 in consecutive blocks.
template <bool NT = true>
__device__ __forceinline__ void load_k_sub(const AttnArgs& a, int lrow, int j, int q, int st, int slot,
                                           q35_u32x4* kf) {
    const int lane = threadIdx.x & 63;
    const int tile = max(min(q * 4 + st, slot >> 4), 0);
    const uint16_t* kp = a.kc + lrow * a.kv_lane + a.kv_layer_off + (size_t)j * a.cap * 256 + (size_t)tile * 4096 + lane * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s)
        kf[s] = NT ? __builtin_nontemporal_load((const q35_u32x4*)(kp + s * 512)) : *(const q35_u32x4*)(kp + s * 512);
}

template <bool NT = true>
__device__ __forceinline__ void load_k_slice(const AttnArgs& a, int lrow, int j, int q, int slot,
                                             q35_u32x4 (*kf)[8]) {
#pragma unroll
    for (int st = 0; st < 4; ++st) load_k_sub<NT>(a, lrow, j, q, st, slot, kf[st]);
}

// Scores of the 64-slot slice q (slots q*64 .. +64, masked beyond `slot`) by one wave.
// Scores -> dst[h * dst_stride + t]; slice stats (max, sum e^(s - max)) ->
// stats[h * stats_stride + 2q .. +1]. No barriers: waves run independently.
// kf holds slice q's K fragments on entry; with REFILL each sub-tile's registers are
// refilled with slice qnext's as soon as its MFMA chain has consumed them (unconditionally:
// past the end every lane reloads row `slot`, so the wait counts stay exact and the loads
// stay in flight across iterations).
template <bool REFILL, bool NT = true>
__device__ __forceinline__ void score_slice(const AttnArgs& a, int lrow, int j, int q, int slot,
                                            const q35_u32x4* qf, q35_u32x4 (*kf)[8], int qnext,
                                            float* dst, size_t dst_stride, float* stats, size_t stats_stride) {
    const int lane = threadIdx.x & 63;
    const int n = lane & 15, g = lane >> 4;
    const int t0 = q * 64;
    float sv[4][4];      // [sub-tile][r] for this lane's head (lanes n < 4)
#pragma unroll
    for (int st = 0; st < 4; ++st) {
        q35_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 8; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[st][s], *(const q35_bf16x8*)&qf[s], acc, 0, 0, 0);
        if (REFILL) load_k_sub<NT>(a, lrow, j, qnext, st, slot, kf[st]);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const float lo = row_down4(acc[rr]);   // lanes n < 4 add the q_lo column n + 4
            const float sc = (acc[rr] + lo) * 0.0625f;
            const int t = t0 + st * 16 + 4 * g + rr;
            const bool ok = n < 4 && t <= slot;
            sv[st][rr] = ok ? sc : -INFINITY;
            if (ok) dst[n * dst_stride + t] = sc;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) m = fmaxf(m, sv[st][rr]);
    m = fmaxf(m, xor16(m));
    m = fmaxf(m, xor32(m));
    float e = 0.f;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) e += sv[st][rr] > -INFINITY ? expf(sv[st][rr] - m) : 0.f;
    e += xor16(e);
    e += xor32(e);
    if (lane < 4 && t0 <= slot) {
        float* sp = stats + lane * stats_stride + 2 * q;
        sp[0] = m;
        sp[1] = e;
    }
}

// q fragments for a one-wave block: lane L converts dims 4L .. 4L+3 of the 4 heads.
__device__ __forceinline__ void load_q_frags_wave(const AttnArgs& a, int r, int j, uint16_t (*qb)[256],
                                                  q35_u32x4* qf) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const float* q = a.q + ((size_t)r * kNq + 4 * j) * 256;
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = 4 * lane + e;
            const float qv = q[h * 256 + d];
            const uint16_t hi = f2bf(qv);
            qb[h][d] = hi;
            qb[4 + h][d] = f2bf(qv - bf2f(hi));
            qb[8 + h][d] = 0;
            qb[12 + h][d] = 0;
        }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const q35_u32x4*)&qb[n][s * 32 + g * 8];
}

// One wave per (row, kv head, 64-slot slice): many small blocks, so a single row's scores
// spread over the CUs.
__global__ void __launch_bounds__(64) attn_scores(AttnArgs a) {
    __shared__ uint16_t qb[16][256];
    const int r = blockIdx.x, j = blockIdx.y, q = blockIdx.z;
    const int slot = a.rm.slot[r];
    if (q * 64 > slot) return;
    q35_u32x4 qf[8], kf[4][8];
    load_k_slice(a, a.rm.lane[r], j, q, slot, kf);
    load_q_frags_wave(a, r, j, qb, qf);
    score_slice<false>(a, a.rm.lane[r], j, q, slot, qf, kf, 0, a.sc + ((size_t)r * kNq + 4 * j) * a.sc_ld, a.sc_ld,
                       a.stats + ((size_t)r * kNq + 4 * j) * a.max_chunks * 8, (size_t)a.max_chunks * 8);
}

// q / k head norm and rope by one wave: lane holds d = lane + 64 w (w = 0..3); the sum of squares
// folds each 64-element quarter with a wave sum and then (q0 + q1) + (q2 + q3).
__device__ __forceinline__ void head_norm_rope_wave(const AttnArgs& a, const uint16_t* src,
                                                    const uint16_t* normw, int pos, float* out) {
    const int lane = threadIdx.x & 63;
    float x[4], ssq[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) x[w] = bf2f(src[lane + 64 * w]);
#pragma unroll
    for (int w = 0; w < 4; ++w) ssq[w] = wave_sum(x[w] * x[w]);
    const float rs = rsqrtf(((ssq[0] + ssq[1]) + (ssq[2] + ssq[3])) * (1.0f / 256.0f) + kEps);
#pragma unroll
    for (int w = 0; w < 4; ++w) out[w] = rbf(__fmul_rn(__fmul_rn(x[w], rs), 1.0f + bf2f(normw[lane + 64 * w])));
    // rope on dims 0..63 (pairs d, d +- 32): quarter 0 holds them, the partner is lane ^ 32
    const float partner = xor32(out[0]);
    const int i = lane & 31;
    const float ang = __fmul_rn((float)pos, a.inv_freq[i]);
    const float c = cosf(ang), sn = sinf(ang);
    const float rot = lane < 32 ? -partner : partner;
    out[0] = __fadd_rn(__fmul_rn(out[0], c), __fmul_rn(rot, sn));
}

// q and new K / V rows of every (row, head), one head per wave: no block barriers, and the rope's
// sine and cosine only where they are used (a 256-thread block per head with two block reductions
// took 8.3 us for 256 rows and 21.6 for 2,048; now 5.8 and 13.3).
__global__ void __launch_bounds__(256) attn_prep(AttnArgs a) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = item / (kNq + kNkv), hh = item % (kNq + kNkv);
    if (r >= a.R) return;
    const uint16_t* pr = a.proj + (size_t)r * kAttnInRows;
    const int pos = a.rm.pos[r];
    float o[4];
    if (hh < kNq) {
        head_norm_rope_wave(a, pr + hh * 512, a.q_norm, pos, o);
#pragma unroll
        for (int w = 0; w < 4; ++w) a.q[((size_t)r * kNq + hh) * 256 + lane + 64 * w] = o[w];
        return;
    }
    const int j = hh - kNq, slot = a.rm.slot[r];
    const size_t base = a.rm.lane[r] * a.kv_lane + a.kv_layer_off + (size_t)j * a.cap * 256;
    uint16_t v[4];                          // before the K stores (see make_kv_row)
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = pr[kAttnVOff + j * 256 + lane + 64 * w];
    head_norm_rope_wave(a, pr + kAttnKOff + j * 256, a.k_norm, pos, o);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int d = lane + 64 * w;
        a.kc[base + kv_tiled_offset(slot, d)] = f2bf(o[w]);
        a.vc[base + kv_v8_offset(slot, d)] = v[w];
    }
}

// A wave's q head into the score operand's columns c (bf16 of q) and c + 4 (its low part). Columns 8 ..
// 15 (of a second row) stay as they are: an MFMA output column depends on its own B column only.
__device__ __forceinline__ void make_q_head(const AttnArgs& a, const uint16_t* src, int pos, uint16_t (*qb)[256], int c) {
    const int lane = threadIdx.x & 63;
    float o[4];
    head_norm_rope_wave(a, src, a.q_norm, pos, o);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int d = lane + 64 * w;
        const uint16_t hi = f2bf(o[w]);
        qb[c][d] = hi;
        qb[4 + c][d] = f2bf(o[w] - bf2f(hi));
    }
}
// A wave's new K row (into the cache and, for the fragments already loaded, knew) and V row. The V
// values are loaded first: behind the K stores, which might alias, each would wait for them.
__device__ __forceinline__ void make_kv_row(const AttnArgs& a, const uint16_t* prow, int pos, int lrow, int j, int slot,
                                            uint16_t* knew) {
    const int lane = threadIdx.x & 63;
    uint16_t v[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = prow[kAttnVOff + j * 256 + lane + 64 * w];
    float o[4];
    head_norm_rope_wave(a, prow + kAttnKOff + j * 256, a.k_norm, pos, o);
    const size_t base = lrow * a.kv_lane + a.kv_layer_off + (size_t)j * a.cap * 256;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int d = lane + 64 * w;
        const uint16_t kb = f2bf(o[w]);
        knew[d] = kb;
        a.kc[base + kv_tiled_offset(slot, d)] = kb;
        a.vc[base + kv_v8_offset(slot, d)] = v[w];
    }
}
// The new K row in place of the fragments of sub-tile st in the lanes that hold its row (selects: with
// a branch around them the compiler indexes the fragments by st and moves them to scratch memory).
__device__ __forceinline__ void patch_k(const uint16_t* knew, int st, int slot, q35_u32x4 (*kf)[8]) {
    const int lane = threadIdx.x & 63;
    const bool mine = (lane & 15) == (slot & 15);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const q35_u32x4 v = *(const q35_u32x4*)&knew[s * 32 + (lane >> 4) * 8];
#pragma unroll
        for (int t = 0; t < 4; ++t) kf[t][s] = mine && t == st ? v : kf[t][s];
    }
}

// The split path with one row per lane (batch-1 decode): attn_prep folded into the slice
// score kernel. Every block makes its 4 q heads itself; the block whose slice holds the new
// slot also makes the new K row, appends K and V to the cache and patches its own K fragments
// for that slot (its global load may still hold the previous contents).
__global__ void __launch_bounds__(64) attn_scores_prep(AttnArgs a) {
    __shared__ uint16_t qb[16][256];
    __shared__ uint16_t knew[256];
    const int r = blockIdx.x, j = blockIdx.y, q = blockIdx.z;
    const int slot = a.rm.slot[r];
    if (q * 64 > slot) return;
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int lrow = a.rm.lane[r], pos = a.rm.pos[r];
    q35_u32x4 qf[8], kf[4][8];
    load_k_slice(a, lrow, j, q, slot, kf);
    const uint16_t* pr = a.proj + (size_t)r * kAttnInRows;
    const bool own = q == (slot >> 6);
#pragma unroll
    for (int i = 0; i < 4; ++i) make_q_head(a, pr + (4 * j + i) * 512, pos, qb, i);
    if (own) make_kv_row(a, pr, pos, lrow, j, slot, knew);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const q35_u32x4*)&qb[n][s * 32 + g * 8];
    if (own) patch_k(knew, (slot >> 4) - q * 4, slot, kf);
    score_slice<false>(a, lrow, j, q, slot, qf, kf, 0, a.sc + ((size_t)r * kNq + 4 * j) * a.sc_ld, a.sc_ld,
                       a.stats + ((size_t)r * kNq + 4 * j) * a.max_chunks * 8, (size_t)a.max_chunks * 8);
}

// P.V over one 128-slot part on MFMA (v_mfma_f32_16x16x32_bf16, k = slots): D = P V with
// A = P (16 query columns x 32 slots: the normalised weights rounded to bf16, from LDS) and
// B = V (32 slots x 16 dims: one 16-byte load of the 8-slot V layout per lane), one chain of
// the part's four 32-slot steps from zero per 16-dim tile; the parts are summed in order.
// Lane (n, g) of D holds query column 4g + r, dim n. A query column's result depends only on
// its own row of P, so one row, a lane's several rows and the split path give the same bits.
// A wave takes 4 dim tiles (64 dims): 16 V fragments per part.
constexpr int kPart = 128;
constexpr int kPlStride = kPart + 8;          // bf16 row stride of P in LDS (conflict-free reads)

// Softmax (max, sum) of the row's 4 heads from the nsl slice stats -> ml[h][0..1]: wave h
// takes head h, lane i folds slices i, i + 64, ... in order, then a fixed xor butterfly.
// Needs 4 waves.
__device__ __forceinline__ void softmax_ml(const float* stats, size_t stats_stride, int nsl, float (*ml)[2]) {
    const int lane = threadIdx.x & 63, h = (threadIdx.x >> 6) & 3;
    const float* st = stats + h * stats_stride;
    float m = -INFINITY;
    for (int i = lane; i < nsl; i += 64) m = fmaxf(m, st[2 * i]);
    m = wave_max(m);
    float l = 0.f;
    for (int i = lane; i < nsl; i += 64) l += st[2 * i + 1] * expf(st[2 * i] - m);
    l = wave_sum(l);
    if (lane == 0) {
        ml[h][0] = m;
        ml[h][1] = l;
    }
}

// V fragments of part pc for dim tiles dt0 .. dt0 + NTL - 1: vf[ks][i] = slots pc*128 + 32 ks +
// 8 g .. +8 of dim 16 (dt0 + i) + n. Unconditional loads with the 8-slot group clamped to slot's
// (past the end every lane re-reads that group, so the wait counts stay exact); slots past
// `slot` are zeroed by mask_vf before use.
template <bool NT = true, int NTL = 4>
__device__ __forceinline__ void load_vf(const AttnArgs& a, int lrow, int j, int pc, int slot, int dt0,
                                        q35_u32x4 (*vf)[NTL]) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const uint16_t* vb = a.vc + lrow * a.kv_lane + a.kv_layer_off + (size_t)j * a.cap * 256;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int sg = min(pc * 16 + 4 * ks + g, slot >> 3);
#pragma unroll
        for (int i = 0; i < NTL; ++i) {
            const q35_u32x4* p = (const q35_u32x4*)(vb + (size_t)sg * 2048 + (16 * (dt0 + i) + n) * 8);
            vf[ks][i] = NT ? __builtin_nontemporal_load(p) : *p;
        }
    }
}

// Zero the V values of slots past `slot` in part pc's fragments (its last part only: V memory
// past the written slots is not initialised, and a zero weight times a NaN would be NaN).
template <int NTL = 4>
__device__ __forceinline__ void mask_vf(int pc, int slot, q35_u32x4 (*vf)[NTL]) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int cnt = slot + 1 - (pc * 128 + 32 * ks + 8 * g);   // valid slots of the group
        uint32_t mk[4];
#pragma unroll
        for (int w = 0; w < 4; ++w)
            mk[w] = (cnt > 2 * w ? 0xffffu : 0u) | (cnt > 2 * w + 1 ? 0xffff0000u : 0u);
#pragma unroll
        for (int i = 0; i < NTL; ++i)
            vf[ks][i] = (q35_u32x4){vf[ks][i][0] & mk[0], vf[ks][i][1] & mk[1], vf[ks][i][2] & mk[2], vf[ks][i][3] & mk[3]};
    }
}

// The part's four 32-slot steps for the wave's NTL dim tiles: out[i] = D of tile dt0 + i.
// pl: P in LDS, [16][kPlStride] bf16 (query column rows); rows >= nq are taken as zero.
template <int NTL = 4>
__device__ __forceinline__ void pv_mfma(const uint16_t* pl, int nq, q35_u32x4 (*vf)[NTL], q35_f32x4* out) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    q35_u32x4 af[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const q35_u32x4 v = *(const q35_u32x4*)(pl + n * kPlStride + 32 * ks + 8 * g);
        af[ks] = n < nq ? v : (q35_u32x4){0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < NTL; ++i) {
        q35_f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&af[ks], *(q35_bf16x8*)&vf[ks][i], d, 0, 0, 0);
        out[i] = d;
    }
}

// A product of a lane's T rows (slots slot_t, ascending) over a part that holds slots past the first
// row's: row t attends up to its own slot, but its zero weight for a later row's slot turns an infinite or
// NaN V there into a NaN. Where a row but the last came out non-finite, rows 0 .. T-2 take products of
// their own with the V past their slot zeroed (a finite V adds nothing there, so a finite product has the
// bits already). Tile by tile, with the masks made again for each: the registers of the parts in flight
// leave no room for more (a whole second product at once moves some of them to scratch memory). Made
// without the check they cost 1 .. 2 us (128 lanes x 3 rows x 2,000 slots: 91 us before, 93.4 so, 91 with it).
template <int T, int NTL>
__device__ __forceinline__ void pv_own_rows(const uint16_t* pl, int pc, const int* slot_t, const q35_u32x4 (*vf)[NTL],
                                            q35_f32x4* out) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int h = 0; h < 4; ++h) top = max(top, __float_as_uint(out[i][h]) & 0x7fffffffu);
    if (!__any(g < T - 1 && top >= 0x7f800000u)) return;
#pragma unroll 1
    for (int t = T - 2; t >= 0; --t) {
        const int left = (t == 0 ? slot_t[0] : slot_t[1]) + 1 - (pc * kPart + 8 * g);
#pragma unroll
        for (int i = 0; i < NTL; ++i) {
            int base = left;                              // a new value to the compiler for each tile
            asm volatile("" : "+v"(base) :: "memory");
            q35_f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const int cnt = base - 32 * ks;           // the row's valid slots of the group (see mask_vf)
                q35_u32x4 af = *(const q35_u32x4*)(pl + n * kPlStride + 32 * ks + 8 * g), v = vf[ks][i];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    af[w] = n < 4 * T ? af[w] : 0u;
                    v[w] &= (cnt > 2 * w ? 0xffffu : 0u) | (cnt > 2 * w + 1 ? 0xffff0000u : 0u);
                }
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&af, *(q35_bf16x8*)&v, d, 0, 0, 0);
            }
#pragma unroll
            for (int h = 0; h < 4; ++h) out[i][h] = g == t ? d[h] : out[i][h];
        }
    }
}

// The weights of part pc for query columns c0 .. c0 + 3 (the 4 heads of one row) into P rows
// c0 .. c0 + 3: p = bf16(e^(s - m) / l), zero past `slot`; `scores` -> head 0's scores of the
// row (head stride s_stride), 256 threads, two weights each.
__device__ __forceinline__ void part_weights(const float* scores, size_t s_stride, const float (*ml)[2], int pc,
                                             int slot, uint16_t* pl, int c0) {
    const int tid = threadIdx.x & 255, t0 = pc * kPart;
    const int nn = min(kPart, slot + 1 - t0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int idx = tid + q * 256, i = idx >> 7, t = idx & 127;
        const float s = t < nn ? scores[i * s_stride + t0 + t] : 0.f;
        pl[(c0 + i) * kPlStride + t] = t < nn ? f2bf(expf(s - ml[i][0]) / ml[i][1]) : (uint16_t)0;
    }
}

// The softmax (max, sum) of a row's 4 heads from its nsl slice stats, in one wave, with
// softmax_ml's arithmetic per head (lane i folds slices i, i + 64, ... in order, then the xor
// butterfly), the heads interleaved so that their loads are in flight together. Every lane
// ends with all four (m, l).
__device__ __forceinline__ void wave_ml(const float* stats, size_t sst, int nsl, float* m, float* l) {
    const int tid = threadIdx.x & 63;
    // slices tid and tid + 64 held in registers (up to 128 slices, an 8,192-slot context),
    // the rest re-read in the second pass; unconditional clamped loads, masked values
#pragma unroll
    for (int h = 0; h < 4; ++h) m[h] = -INFINITY;
    float sm0[4][2], se0[4][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = min(tid + 64 * u, nsl - 1);
        const bool ok = tid + 64 * u < nsl;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const float2 v = *(const float2*)(stats + h * sst + 2 * i);
            sm0[h][u] = ok ? v.x : -INFINITY;
            se0[h][u] = v.y;
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int h = 0; h < 4; ++h) m[h] = fmaxf(m[h], sm0[h][u]);
    for (int i = tid + 128; i < nsl; i += 64) {
#pragma unroll
        for (int h = 0; h < 4; ++h) m[h] = fmaxf(m[h], stats[h * sst + 2 * i]);
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) m[h] = wave_max(m[h]);
#pragma unroll
    for (int h = 0; h < 4; ++h) l[h] = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (tid + 64 * u < nsl) {
#pragma unroll
            for (int h = 0; h < 4; ++h) l[h] += se0[h][u] * expf(sm0[h][u] - m[h]);
        }
    for (int i = tid + 128; i < nsl; i += 64) {
        float sm[4], se[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) { sm[h] = stats[h * sst + 2 * i]; se[h] = stats[h * sst + 2 * i + 1]; }
#pragma unroll
        for (int h = 0; h < 4; ++h) l[h] += se[h] * expf(sm[h] - m[h]);
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) l[h] = wave_sum(l[h]);
}

// A row's outputs bf16(bf16(sum of parts) * bf16(sigmoid(gate))) for the 4 heads of kv group j and
// dims d0 + 16 i (acc[i][h]): every gate is loaded before the first store (a gate load behind a
// store waits for it -- they might alias -- and 8 or 16 round trips then end the block).
template <int NTL>
__device__ __forceinline__ void store_gated(const AttnArgs& a, int r, int j, int d0, const q35_f32x4* acc) {
    const uint16_t* pr = a.proj + (size_t)r * kAttnInRows + 4 * j * 512 + 256 + d0;
    uint16_t* po = a.out + (size_t)r * 2048 + 4 * j * 256 + d0;
    uint16_t graw[NTL][4];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int h = 0; h < 4; ++h) graw[i][h] = pr[h * 512 + 16 * i];
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int h = 0; h < 4; ++h)
            po[h * 256 + 16 * i] = f2bf(rbf(acc[i][h]) * rbf(sigmoid_f(bf2f(graw[i][h]))));
}

// A part's partial sums: [row][part][kv head][dim][4 heads], so a lane's four heads of one dim
// (one MFMA accumulator) are one 16-byte store.
__device__ __forceinline__ size_t part_offset(const AttnArgs& a, int r, int pc, int j, int d) {
    return ((((size_t)r * a.max_chunks * 2 + pc) * kNkv + j) * 256 + d) * 4;
}

// Split path, one block per (row, kv head, part): wave w takes dims 64w .. +64.
__global__ void __launch_bounds__(256) attn_pv(AttnArgs a) {
    __shared__ uint16_t pl[16 * kPlStride];
    __shared__ float ml[4][2];
    const int r = blockIdx.x, j = blockIdx.y, pc = blockIdx.z;
    const int slot = a.rm.slot[r];
    if (pc >= slot / kPart + 1) return;
    const int lrow = a.rm.lane[r], wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    q35_u32x4 vf[4][4];
    load_vf(a, lrow, j, pc, slot, 4 * wv, vf);
    softmax_ml(a.stats + ((size_t)r * kNq + 4 * j) * a.max_chunks * 8, (size_t)a.max_chunks * 8, slot / 64 + 1, ml);
    __syncthreads();
    part_weights(a.sc + ((size_t)r * kNq + 4 * j) * a.sc_ld, a.sc_ld, ml, pc, slot, pl, 0);
    __syncthreads();
    if (pc == slot / kPart) mask_vf(pc, slot, vf);
    q35_f32x4 out[4];
    pv_mfma(pl, 4, vf, out);
    if (lane < 16) {
        float* pp = a.part + part_offset(a, r, pc, j, 64 * wv + lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) *(q35_f32x4*)(pp + 64 * i) = out[i];
    }
}

// Sum of the 128-slot partials in part order, bf16, times bf16(sigmoid(gate)). Block (row, kv
// head, 64 dims), a thread per (dim, head). whole: the most parts of a lane whose pairs
// attn_seg_pv finishes by itself (its T rows' last slot decides; 0: none).
__global__ void __launch_bounds__(256) attn_combine(AttnArgs a, int whole) {
    const int r = blockIdx.x, j = blockIdx.y >> 2, tid = threadIdx.x, h = tid & 3;
    const int d = (blockIdx.y & 3) * 64 + (tid >> 2);
    const int nparts = a.rm.slot[r] / kPart + 1;
    if (whole) {
        int last = 0;
        for (int t = 0, r0 = r / a.T * a.T; t < a.T; ++t) last = max(last, a.rm.slot[r0 + t]);
        if (last / kPart + 1 <= whole) return;
    }
    const float* pp = a.part + part_offset(a, r, 0, j, d) + h;
    const uint16_t graw = a.proj[(size_t)r * kAttnInRows + (4 * j + h) * 512 + 256 + d];
    float acc = 0.f;
    // 40 parts per round (a 5,120-slot context in one), all loads issued before the adds:
    // unconditional from clamped part indices, so no branch makes the compiler wait per load
    for (int c0 = 0; c0 < nparts; c0 += 40) {
        float v[40];
#pragma unroll
        for (int u = 0; u < 40; ++u) v[u] = pp[(size_t)min(c0 + u, nparts - 1) * kNq * 256];
#pragma unroll
        for (int u = 0; u < 40; ++u)
            if (c0 + u < nparts) acc += v[u];
    }
    const float o = rbf(acc);
    const float g = rbf(sigmoid_f(bf2f(graw)));
    a.out[(size_t)r * 2048 + (4 * j + h) * 256 + d] = f2bf(o * g);
}

// ---------------------------------------------------------------- split path, 4-wave blocks
// The split path's kernels with more waves per block and the same arithmetic, so a row's
// K/V streams over 4x the waves (batch 1 uses a quarter of the CUs otherwise):
//   attn_scores4   (row, kv head, 64-slot slice): wave w scores 16-slot sub-tile w (8 KiB of
//                  K) and, with PREP, makes q head 4j + w (wave 0 also the new K row); wave 0
//                  then forms the slice stats from all four sub-tiles' values in score_slice's
//                  order (max, then e summed sub-tile-major)
//   attn_pv4       (row, kv head, 128-slot part, 64-dim quarter): one wave, the part's P.V
//                  for its 4 dim tiles on MFMA (pv_mfma), the weights made in the wave
template <bool PREP>
__global__ void __launch_bounds__(256) attn_scores4(AttnArgs a) {
    __shared__ uint16_t qb[16][256];
    __shared__ uint16_t knew[256];
    __shared__ float svl[4][4][64];          // [sub-tile][r][lane]
    const int r = blockIdx.x, j = blockIdx.y, q = blockIdx.z;
    const int slot = a.rm.slot[r];
    if (q * 64 > slot) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n = lane & 15, g = lane >> 4;
    const int lrow = a.rm.lane[r];
    q35_u32x4 qf[8], kf[8];
    load_k_sub(a, lrow, j, q, wv, slot, kf);
    const bool own = PREP && q == (slot >> 6);
    if (PREP) {
        const int pos = a.rm.pos[r];
        const uint16_t* pr = a.proj + (size_t)r * kAttnInRows;
        make_q_head(a, pr + (4 * j + wv) * 512, pos, qb, wv);
        if (own && wv == 0) make_kv_row(a, pr, pos, lrow, j, slot, knew);
    } else {
        const float* qp = a.q + ((size_t)r * kNq + 4 * j + wv) * 256;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int d = lane + 64 * w;
            const float qv = qp[d];
            const uint16_t hi = f2bf(qv);
            qb[wv][d] = hi;
            qb[4 + wv][d] = f2bf(qv - bf2f(hi));
            qb[8 + wv][d] = 0;
            qb[12 + wv][d] = 0;
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const q35_u32x4*)&qb[n][s * 32 + g * 8];
    if (own && n == (slot & 15) && wv == (slot >> 4) - q * 4) {
#pragma unroll
        for (int s = 0; s < 8; ++s) kf[s] = *(const q35_u32x4*)&knew[s * 32 + g * 8];
    }
    float* dst = a.sc + ((size_t)r * kNq + 4 * j) * a.sc_ld;
    const int t0 = q * 64;
    {
        q35_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 8; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[s], *(const q35_bf16x8*)&qf[s], acc, 0, 0, 0);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            const float lo = row_down4(acc[rr]);   // lanes n < 4 add the q_lo column n + 4
            const float sc = (acc[rr] + lo) * 0.0625f;
            const int t = t0 + wv * 16 + 4 * g + rr;
            const bool ok = n < 4 && t <= slot;
            svl[wv][rr][lane] = ok ? sc : -INFINITY;
            if (ok) dst[n * a.sc_ld + t] = sc;
        }
    }
    __syncthreads();
    if (wv != 0) return;
    float sv[4][4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) sv[st][rr] = svl[st][rr][lane];
    float m = -INFINITY;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) m = fmaxf(m, sv[st][rr]);
    m = fmaxf(m, xor16(m));
    m = fmaxf(m, xor32(m));
    float e = 0.f;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) e += sv[st][rr] > -INFINITY ? expf(sv[st][rr] - m) : 0.f;
    e += xor16(e);
    e += xor32(e);
    if (lane < 4) {
        float* sp = a.stats + ((size_t)r * kNq + 4 * j + lane) * a.max_chunks * 8 + 2 * q;
        sp[0] = m;
        sp[1] = e;
    }
}

__global__ void __launch_bounds__(64) attn_pv4(AttnArgs a) {
    __shared__ uint16_t pl[16 * kPlStride];
    const int r = blockIdx.x, j = blockIdx.y, pc = blockIdx.z >> 2, dq = blockIdx.z & 3;
    const int slot = a.rm.slot[r];
    if (pc >= slot / kPart + 1) return;
    const int tid = threadIdx.x;
    const int lrow = a.rm.lane[r];
    const int t0 = pc * kPart;
    // V fragments first (unconditional clamped loads), as load_vf does
    q35_u32x4 vf[4][4];
    load_vf(a, lrow, j, pc, slot, 4 * dq, vf);
    // this part's raw scores (independent of the softmax statistics: loaded early)
    const int n = min(kPart, slot + 1 - t0);
    const float* scores = a.sc + ((size_t)r * kNq + 4 * j) * a.sc_ld;
    float sraw[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int idx = tid + k * 64, i = idx >> 7, t = idx & 127;
        sraw[k] = scores[i * a.sc_ld + t0 + min(t, n - 1)];
    }
    float m[4], l[4];
    wave_ml(a.stats + ((size_t)r * kNq + 4 * j) * a.max_chunks * 8, (size_t)a.max_chunks * 8, slot / 64 + 1, m, l);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int idx = tid + k * 64, i = idx >> 7, t = idx & 127;
        const float mi = i == 0 ? m[0] : i == 1 ? m[1] : i == 2 ? m[2] : m[3];
        const float li = i == 0 ? l[0] : i == 1 ? l[1] : i == 2 ? l[2] : l[3];
        pl[i * kPlStride + t] = t < n ? f2bf(expf(sraw[k] - mi) / li) : (uint16_t)0;
    }
    __syncthreads();
    if (pc == slot / kPart) mask_vf(pc, slot, vf);
    q35_f32x4 out[4];
    pv_mfma(pl, 4, vf, out);
    if (tid < 16) {
        float* pp = a.part + part_offset(a, r, pc, j, dq * 64 + tid);
#pragma unroll
        for (int i = 0; i < 4; ++i) *(q35_f32x4*)(pp + 64 * i) = out[i];
    }
}

// Batched lanes: one block per (row, kv head) runs every chunk's scores into LDS, the
// softmax, every part's P.V and the gated sum -- the same device functions and orders as the
// split kernels, without the score / stats / partial round trips through HBM.
// NI = 2 (one row per lane): a block of 512 threads runs two (row, kv head) items, one per
// 256-thread half, with their own LDS. Two one-item blocks sharing a CU do not progress
// evenly (the older block's waves win the issue arbitration: at 256 lanes and ctx 4096 the
// first-dispatched half of the grid finished at ~260 us and the other at ~330 us, the CUs
// half idle in between); the halves of one block meet at every barrier, so both items end
// together. A half with fewer parts runs idle parts (its loads clamped, its sums not added)
// to keep the barrier count equal.
// PREP (one row per lane, no lane twice): the item's q heads and its new K / V row are made here, by
// wave (q head wv; wave 0 also the K row, into the q staging's unused column 8), instead of by
// attn_prep (8 us and a launch gap at 256 rows); the K fragments of the new slot, loaded before it
// was written, are patched from there.
template <bool NT, int NI, bool PREP>
__global__ void __launch_bounds__(256 * NI) attn_fused(AttnArgs a, int lds_slots) {
    extern __shared__ float fl[];
    const int half = NI == 1 ? 0 : (int)(threadIdx.x >> 8);
    const size_t item_lds = (size_t)4 * lds_slots + (size_t)4 * 8 * a.max_chunks;
    float* scl = fl + half * item_lds;                  // [4][lds_slots]
    float* stl = scl + 4 * lds_slots;                   // [4][8 * max_chunks]
    __shared__ float ubuf_all[NI][2048];                // q staging, then the part's weights
    __shared__ float ml_all[NI][4][2];
    __shared__ int nparts_all[NI];
    uint16_t(*qb)[256] = (uint16_t(*)[256])ubuf_all[half];
    float(*ml)[2] = ml_all[half];
    // Block order: the T rows of one lane read the same K/V, so they run as consecutive
    // blocks of one XCD (blocks go round-robin to the 8 XCDs) and share its L2 stream. With
    // fewer (lane, kv head) pairs than XCDs (a prompt wave of one lane) each pair's rows are
    // cut into `nseg` contiguous segments of `seg` rows so that every XCD gets a segment:
    // virtual pair v -> XCD v % 8, blocks 8 ((v / 8) seg + i) + v % 8. With NI = 2 the
    // virtual blocks 16 (b / 8) + b % 8 and that + 8 run in block b (same XCD).
    const int T = a.T, tid = threadIdx.x & 255;
    const int npairs = (a.R / T) * kNkv;
    const int nseg = max(1, 8 / npairs), seg = (T + nseg - 1) / nseg;
    const int vb = NI == 1 ? (int)blockIdx.x : (int)(blockIdx.x >> 3) * 16 + half * 8 + (int)(blockIdx.x & 7);
    const int xcd = vb & 7, kk = vb >> 3;
    const int v = (kk / seg) * 8 + xcd;
    const int pr = v / nseg, t = (v % nseg) * seg + kk % seg;
    const bool active = v < npairs * nseg && t < T;
    if (NI == 1 && !active) return;
    const int j = pr % kNkv, r = active ? (pr / kNkv) * T + t : 0;
    const int slot = active ? a.rm.slot[r] : 0;
    const int lrow = a.rm.lane[r];
    const int nch = active ? slot / kChunk + 1 : 0, nparts = active ? slot / kPart + 1 : 0;
    const size_t sst = (size_t)a.max_chunks * 8;
    q35_u32x4 qf[8];
    {
        const int wv = tid >> 6;
        q35_u32x4 kf[4][8];
        load_k_slice<NT>(a, lrow, j, wv, slot, kf);
        if constexpr (PREP) {
            const int lane = tid & 63, n = lane & 15, g = lane >> 4;
            const uint16_t* prow = a.proj + (size_t)r * kAttnInRows;
            const int pos = a.rm.pos[r];
            make_q_head(a, prow + (4 * j + wv) * 512, pos, qb, wv);
            if (wv == 0 && active) make_kv_row(a, prow, pos, lrow, j, slot, qb[8]);
            __syncthreads();
#pragma unroll
            for (int s = 0; s < 8; ++s) qf[s] = *(const q35_u32x4*)&qb[n][s * 32 + g * 8];
        } else {
            load_q_frags(a, r, j, qb, qf);
        }
        // wave wv takes slices 4c + wv; the last one refills nothing (no loads past the end
        // ahead of the V stream's first loads)
        for (int c = 0; c + 1 < nch; ++c)
            score_slice<true, NT>(a, lrow, j, 4 * c + wv, slot, qf, kf, 4 * (c + 1) + wv, scl, lds_slots, stl, sst);
        if (PREP && nch > 0 && (slot >> 6) == 4 * (nch - 1) + wv) patch_k(qb[8], (slot >> 4) & 3, slot, kf);
        if (nch > 0) score_slice<false, NT>(a, lrow, j, 4 * (nch - 1) + wv, slot, qf, kf, 0, scl, lds_slots, stl, sst);
    }
    if (NI > 1 && tid == 0) nparts_all[half] = nparts;
    __syncthreads();
    int np = nparts;
    if (NI > 1) np = max(nparts_all[0], nparts_all[NI - 1]);
    // P.V: wave wv takes dims 64 wv .. +64 (pv_mfma); each part's V fragments are refilled
    // with the next part's right after their MFMAs and stay in flight across the LDS-only
    // barriers. The q staging holds the part's weights.
    const int wv = tid >> 6, lane = tid & 63;
    uint16_t* pl = (uint16_t*)ubuf_all[half];
    // V two parts ahead (the K registers of the score pass are free here): parts alternate
    // between vfa and vfb, each refilled with the part after next once used; a part at np
    // (np odd) is idle like a short half's parts: zero weights, its sum not added
    q35_u32x4 vfa[4][4], vfb[4][4];
    load_vf<NT>(a, lrow, j, 0, slot, 4 * wv, vfa);
    load_vf<NT>(a, lrow, j, 1, slot, 4 * wv, vfb);
    softmax_ml(stl, sst, slot / 64 + 1, ml);
    q35_f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
    auto part = [&](int pc, q35_u32x4 (&vf)[4][4]) {
        lds_barrier();          // ml is in; every wave is done with the previous part's weights
        part_weights(scl, lds_slots, ml, pc, slot, pl, 0);
        lds_barrier();
        if (pc == nparts - 1) mask_vf(pc, slot, vf);
        q35_f32x4 out[4];
        pv_mfma(pl, 4, vf, out);
        load_vf<NT>(a, lrow, j, pc + 2, slot, 4 * wv, vf);
        if (pc < nparts) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += out[i];
        }
    };
    for (int pc = 0; pc < np; pc += 2) {
        part(pc, vfa);
        part(pc + 1, vfb);
    }
    if (active && lane < 16) store_gated<4>(a, r, j, 64 * wv + lane, acc);
}

// MTP verify rows at many lanes (T = 2 or 3 rows per lane at consecutive slots): one block
// per (lane, kv head) for all T rows, so the lane's K/V stream from HBM once and through the
// block once (one block per row re-read each line from L2 three times: ~45 GB/s per CU of
// L2 -> CU traffic for the same HBM rate). Every K fragment feeds the score MFMAs of all T
// rows: B tile u holds rows 2u and 2u + 1 as columns 8 (t % 2) + h (q hi) and + 4 (q lo), and
// an MFMA output column depends only on its own B column, so a row's scores and slice stats
// are the one-row kernel's bits. Each V part, loaded once into registers, feeds the P.V of
// every row at once (the rows' weights are rows of P). T rows x 4 heads x cap f32 scores do
// not fit LDS beside two blocks per CU: the last kRowsLdsParts parts' scores stay in LDS (the
// first written, the last read), the rest go to the global scratch; the block reads back only
// what it wrote, after a block barrier.
// W = 8 (engine option attn_rows 2): one block of 8 waves per CU -- the memory parallelism of
// two 4-wave blocks, and three times the LDS tail; P.V then takes 2 dim tiles per wave.
// PREP (no lane twice): q and the T new K / V rows made here, one head per wave and turn, instead of
// by attn_prep; the K fragments of the new slots are patched from LDS where they are used.
template <int T, int W, bool PREP>
__global__ void __launch_bounds__(64 * W) attn_rows(AttnArgs a) {
    extern __shared__ float stl_all[];                  // [T][4][8 * max_chunks] slice stats, then
                                                        // the LDS tail [T][4][lpn * 128]
    __shared__ uint16_t qbuf[2][16][256];               // q staging (tiles), then the part's weights
    __shared__ float ml_all[T][4][2];
    constexpr int NU = (T + 1) / 2;                     // q tiles
    constexpr int NTL = 16 / W;                         // P.V dim tiles per wave
    constexpr int WPT = 8 / W;                          // weights per thread and row of a part
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n = lane & 15, g = lane >> 4;
    const int pr = blockIdx.x, j = pr % kNkv, r0 = (pr / kNkv) * T;
    int slot_t[T];
#pragma unroll
    for (int t = 0; t < T; ++t) slot_t[t] = a.rm.slot[r0 + t];
    int slot = slot_t[0];
#pragma unroll
    for (int t = 1; t < T; ++t) slot = max(slot, slot_t[t]);
    const int lrow = a.rm.lane[r0];
    const size_t sst = (size_t)a.max_chunks * 8;
    float* tl = stl_all + (size_t)T * 4 * sst;
    const int lpn = rows_lds_parts(T, a.max_chunks, W), lsl = 128 * lpn;
    const int p0 = max(slot / kPart + 1 - lpn, 0);     // first part in the LDS tail
    // q fragments: tile u, column 8 (t % 2) + h = bf16(q) of row t = 2u + t % 2, head h, and
    // + 4 its low part (zero columns for a missing row), as load_q_frags makes them
    // the new K rows, in the columns of q tile 1 that no row has
    uint16_t(*knew)[256] = &qbuf[1][8];
    q35_u32x4 kf[2][8];
    const int nch = (slot / 64 + W) / W;                 // rounds of W slices
    // K two sub-tiles ahead (kf[st % 2] holds sub-tile st; the registers of sub-tile st are refilled
    // with sub-tile st + 2, then the next slice's); the first slice's sub-tile 0 strictly before its
    // sub-tile 1: the loop head's wait for sub-tile 0 must hold on entry too, and with sub-tile 0
    // loaded last it would drain the whole prefetch (and the previous slice's score stores) at
    // every slice
    load_k_sub<true>(a, lrow, j, W * (nch - 1) + wv, 0, slot, kf[0]);
    __builtin_amdgcn_sched_barrier(0);
    load_k_sub<true>(a, lrow, j, W * (nch - 1) + wv, 1, slot, kf[1]);
    if constexpr (PREP) {
        // heads 0 .. 4T-1: q of (row, head); 4T .. 5T-1: the new K row of row i - 4T
        for (int i = __builtin_amdgcn_readfirstlane(wv); i < 5 * T; i += W) {
            const int t = i < 4 * T ? i >> 2 : i - 4 * T;
            const uint16_t* prow = a.proj + (size_t)(r0 + t) * kAttnInRows;
            const int pos = a.rm.pos[r0 + t];
            if (i >= 4 * T) {
                make_kv_row(a, prow, pos, lrow, j, a.rm.slot[r0 + t], knew[t]);
                continue;
            }
            float o[4];
            head_norm_rope_wave(a, prow + (4 * j + (i & 3)) * 512, a.q_norm, pos, o);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint16_t hi = f2bf(o[w]);
                qbuf[t >> 1][8 * (t & 1) + (i & 3)][lane + 64 * w] = hi;
                qbuf[t >> 1][8 * (t & 1) + (i & 3) + 4][lane + 64 * w] = f2bf(o[w] - bf2f(hi));
            }
        }
    } else
    if (tid < 256) {
#pragma unroll
        for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int c = 8 * (t & 1) + h;
                if (t < T) {
                    const float qv = a.q[((size_t)(r0 + t) * kNq + 4 * j + h) * 256 + tid];
                    const uint16_t hi = f2bf(qv);
                    qbuf[t >> 1][c][tid] = hi;
                    qbuf[t >> 1][c + 4][tid] = f2bf(qv - bf2f(hi));
                } else {
                    qbuf[t >> 1][c][tid] = 0;
                    qbuf[t >> 1][c + 4][tid] = 0;
                }
            }
    }
    __syncthreads();
    int smin = slot_t[0];
#pragma unroll
    for (int t = 1; t < T; ++t) smin = min(smin, slot_t[t]);
    // scores: wave wv takes slices W c + wv (score_slice's arithmetic, one MFMA chain per tile)
    {
        q35_u32x4 qf[NU][8];
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int s = 0; s < 8; ++s) qf[u][s] = *(const q35_u32x4*)&qbuf[u][n][s * 32 + g * 8];
        // this block's rows of the score scratch as a buffer resource (byte offsets)
        const __amdgpu_buffer_rsrc_t scres = __builtin_amdgcn_make_buffer_rsrc(
            (void*)uniform_ptr((const char*)(a.sc + (size_t)r0 * kNq * a.sc_ld)), 0, T * kNq * a.sc_ld * 4, 0x00020000);
        const int tr = n >> 3;                           // this lane's row within a tile: 2u + tr
        int lslot[NU];                                   // that row's slot (-1: no such row)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int ta = 2 * u, tb = 2 * u + 1 < T ? 2 * u + 1 : 2 * u;
            lslot[u] = tr == 0 ? slot_t[ta] : 2 * u + 1 < T ? slot_t[tb] : -1;
        }
        // chunks from the last down (a slice's scores and stats do not depend on the order):
        // the top parts, written first, stay in the LDS tail, and the P.V pass starts on the
        // scores written last, still in L2
        for (int c = nch - 1; c >= 0; --c) {
            const int q = W * c + wv, qnext = W * (c - 1) + wv, t0 = q * 64;
            const bool inl = q >= 2 * p0;                // this slice's scores go to the LDS tail
            float sv[NU][4][4];
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                if (PREP && 4 * q + st >= smin >> 4) {   // new K rows: their loads may be stale
#pragma unroll
                    for (int t = 0; t < T; ++t)
                        if (slot_t[t] >> 4 == 4 * q + st && n == (slot_t[t] & 15)) {
#pragma unroll
                            for (int s = 0; s < 8; ++s) kf[st & 1][s] = *(const q35_u32x4*)&knew[t][s * 32 + g * 8];
                        }
                }
                q35_f32x4 acc[NU];
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    acc[u] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 8; ++s)
                        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[st & 1][s], *(const q35_bf16x8*)&qf[u][s], acc[u], 0, 0, 0);
                }
                if (st < 2) load_k_sub<true>(a, lrow, j, q, st + 2, slot, kf[st & 1]);
                else load_k_sub<true>(a, lrow, j, qnext, st - 2, slot, kf[st & 1]);
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    // the lane's 4 consecutive slots go out as one 16-byte store (slots past the
                    // row's last are never read: the P.V pass gives them zero weight)
                    q35_f32x4 scv;
                    const int t = 2 * u + tr, tt0 = t0 + st * 16 + 4 * g;
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const float lo = row_down4(acc[u][rr]);   // lanes with n % 8 < 4 add the q_lo column
                        const float sc = (acc[u][rr] + lo) * 0.0625f;
                        const bool ok = (n & 7) < 4 && tt0 + rr <= lslot[u];
                        sv[u][st][rr] = ok ? sc : -INFINITY;
                        scv[rr] = sc;
                    }
                    // slices below the LDS tail: an unconditional buffer store (lanes without a
                    // score get an offset past the range, which the hardware drops; a store
                    // under a branch would make the compiler drain outstanding loads at the join)
                    const bool okst = (n & 7) < 4 && tt0 <= lslot[u] && !inl;
                    const int off = okst ? ((t * kNq + 4 * j + (n & 3)) * a.sc_ld + tt0) * 4 : 0x7ffffff0;
                    __builtin_amdgcn_raw_buffer_store_b128(
                        (q35_u32x4){__float_as_uint(scv[0]), __float_as_uint(scv[1]), __float_as_uint(scv[2]), __float_as_uint(scv[3])},
                        scres, off, 0, 0);
                    if (inl && (n & 7) < 4 && tt0 <= lslot[u])
                        *(q35_f32x4*)(tl + (t * 4 + (n & 3)) * lsl + (tt0 - 128 * p0)) = scv;
                }
                // sub-tiles stay in order: with the next sub-tile's MFMAs hoisted into this one
                // their K wait also drained this slice's earlier score stores
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                float m = -INFINITY;
#pragma unroll
                for (int st = 0; st < 4; ++st)
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) m = fmaxf(m, sv[u][st][rr]);
                m = fmaxf(m, xor16(m));
                m = fmaxf(m, xor32(m));
                float e = 0.f;
#pragma unroll
                for (int st = 0; st < 4; ++st)
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) e += sv[u][st][rr] > -INFINITY ? expf(sv[u][st][rr] - m) : 0.f;
                e += xor16(e);
                e += xor32(e);
                const int t = 2 * u + tr;
                if (g == 0 && (n & 7) < 4 && t0 <= lslot[u]) {
                    float* sp = stl_all + ((size_t)t * 4 + (n & 3)) * sst + 2 * q;
                    sp[0] = m;
                    sp[1] = e;
                }
            }
        }
    }
    __syncthreads();          // scores (global scratch) and stats (LDS) of every wave are in
#pragma unroll
    for (int t = 0; t < T; ++t) softmax_ml(stl_all + (size_t)t * 4 * sst, sst, slot_t[t] / 64 + 1, ml_all[t]);
    // P.V: P rows 4t + h hold row t's weights, so one pv_mfma per part serves every row (a
    // query column's result depends only on its own weights: the one-row kernel's bits);
    // the q staging holds the weights
    uint16_t* pl = &qbuf[0][0][0];
    // V two parts ahead (the K and q registers of the score pass are free here): parts
    // alternate between vfa and vfb, each refilled with the part after next once used
    q35_f32x4 acc[NTL];
#pragma unroll
    for (int i = 0; i < NTL; ++i) acc[i] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
    const int np = slot / kPart + 1, pown = (smin + 1) / kPart;   // parts from pown on hold slots past the first row's
    // the thread's scores (head i = idx / 128, slot idx % 128 of the part, idx = tid + 64 W q)
    // of every row, loaded two parts ahead like V and issued just before that part's V
    // (clamped to the last slot: unconditional). The vector-memory counter completes in
    // order, so waiting for a part's scores then never waits for V loads issued later.
    // Both sources without a branch, chosen where they are used (a part in the LDS tail reads slot
    // 0 of the scratch, one line for every lane; chosen here, the scratch load would be waited for
    // a part after its issue).
    struct Scores { float gv[T][WPT], lv[T][WPT]; };
    auto load_scores = [&](int pc, Scores& sr) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < WPT; ++q) {
                const int idx = tid + q * 64 * W, i = idx >> 7, tt = idx & 127;
                const int ts = min(pc * kPart + tt, slot);
                const bool lp = pc >= p0 && lpn > 0;
                sr.gv[t][q] = a.sc[((size_t)(r0 + t) * kNq + 4 * j + i) * a.sc_ld + (lp ? 0 : ts)];
                sr.lv[t][q] = *(lp ? tl + (t * 4 + i) * lsl + max(ts - 128 * p0, 0) : stl_all);
            }
    };
    q35_u32x4 vfa[4][NTL], vfb[4][NTL];
    Scores sra, srb;
    // in this order (the loop's waits must hold on entry as well: with a part's scores issued
    // after its V, the first wait of every part would drain the whole V prefetch)
    load_scores(0, sra);
    __builtin_amdgcn_sched_barrier(0);
    load_vf<true, NTL>(a, lrow, j, 0, slot, NTL * wv, vfa);
    __builtin_amdgcn_sched_barrier(0);
    load_scores(1, srb);
    __builtin_amdgcn_sched_barrier(0);
    load_vf<true, NTL>(a, lrow, j, 1, slot, NTL * wv, vfb);
    __builtin_amdgcn_sched_barrier(0);
    const int tg = lane >> 4;
    const int myslot = tg == 0 ? slot_t[0] : tg == 1 ? slot_t[T > 1 ? 1 : 0] : slot_t[T > 2 ? 2 : 0];
    // one part (a part at np, when np is odd, is idle: zero weights, its sum not added)
    auto part = [&](int pc, q35_u32x4 (&vf)[4][NTL], Scores& sr) {
        const bool lp = pc >= p0 && lpn > 0;
        lds_barrier();          // ml is in; every wave is done with the previous part's weights
        // part_weights' arithmetic, from the scores in registers
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int nn = min(kPart, slot_t[t] + 1 - pc * kPart);
#pragma unroll
            for (int q = 0; q < WPT; ++q) {
                const int idx = tid + q * 64 * W, i = idx >> 7, tt = idx & 127;
                const float sc = lp ? sr.lv[t][q] : sr.gv[t][q];
                pl[(4 * t + i) * kPlStride + tt] = tt < nn ? f2bf(expf(sc - ml_all[t][i][0]) / ml_all[t][i][1]) : (uint16_t)0;
            }
        }
        lds_barrier();
        if (pc == np - 1) mask_vf<NTL>(pc, slot, vf);
        q35_f32x4 out[NTL];
        pv_mfma<NTL>(pl, 4 * T, vf, out);
        if (pc >= pown) pv_own_rows<T, NTL>(pl, pc, slot_t, vf, out);
        load_scores(pc + 2, sr);
        load_vf<true, NTL>(a, lrow, j, pc + 2, slot, NTL * wv, vf);
        // lane (n, g) holds row g's heads: add this part where it is one of that row's parts
        if (tg < T && pc < myslot / kPart + 1) {
#pragma unroll
            for (int i = 0; i < NTL; ++i) acc[i] += out[i];
        }
    };
    for (int pc = 0; pc < np; pc += 2) {
        part(pc, vfa, sra);
        part(pc + 1, vfb, srb);
    }
    if (tg < T) store_gated<NTL>(a, r0 + tg, j, 16 * NTL * wv + (lane & 15), acc);
}

// ---------------------------------------------------------------- verify rows by segments
// T = 2 or 3 rows of a lane at few lanes, or at many of which a few are long: the lane's K/V stream once
// for all of its rows, as in attn_rows, but cut into segments of a (lane, kv head) pair, so that a few
// long contexts fill the CUs (the split path's blocks take one row each and read the K/V T times):
//   attn_seg_scores  (pair, 256-slot chunk): wave w scores slice w of the chunk for every row; q
//                    and, with PREP, the chunk's new K / V rows are made by the block; scores and
//                    slice stats leave as whole lines
//   attn_seg_pv      (pair, kSegParts parts): attn_rows' P.V over the segment's parts; a pair of one
//                    segment is finished here, longer ones leave their parts to attn_combine
// Slices, parts and their sums are the other forms', so the results are the same bits. Bound by
// the K/V stream plus the scores' and parts' round trip (a tenth of its bytes, but a fifth of the
// time: writes between the reads cost HBM several times their size). us, split path -> segments:
// 24 lanes x 3 rows x 8,192 slots 277 -> 127, ragged 178 -> 100; 16 x 3 x 2,000 65 -> 50.
constexpr int kSegRow = 68;                              // floats of a slice's (row, head) in LDS: 64 scores, max, sum
constexpr int kSegParts = 4;                             // parts (128 slots) of a P.V segment

// Block -> (pair, segment): a pair's segments in consecutive blocks of one XCD, so that lanes of
// different lengths load the XCDs alike.
__device__ __forceinline__ bool seg_of(const AttnArgs& a, int nseg, int& pr, int& seg) {
    const int k = blockIdx.x >> 3;
    pr = (k / nseg) * 8 + (blockIdx.x & 7);
    seg = k % nseg;
    return pr < a.R / a.T * kNkv;
}

template <int T, bool PREP>
__global__ void __launch_bounds__(256, 2) attn_seg_scores(AttnArgs a, int nseg) {
    constexpr int NU = (T + 1) / 2;                     // q tiles
    __shared__ uint16_t qbuf[NU][16][256];
    __shared__ uint16_t knew[T][256];
    __shared__ float ss_all[4][T][4][kSegRow];          // each wave's slice, then whole lines to memory
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n = lane & 15, g = lane >> 4;
    int pr, c;
    if (!seg_of(a, nseg, pr, c)) return;
    const int j = pr % kNkv, r0 = (pr / kNkv) * T;
    int slot_t[T];
#pragma unroll
    for (int t = 0; t < T; ++t) slot_t[t] = a.rm.slot[r0 + t];
    int slot = slot_t[0];
#pragma unroll
    for (int t = 1; t < T; ++t) slot = max(slot, slot_t[t]);
    if (c * kChunk > slot) return;
    const int lrow = a.rm.lane[r0], q = 4 * c + wv, t0 = q * 64;
    q35_u32x4 kf[2][8];
    load_k_sub<true>(a, lrow, j, q, 0, slot, kf[0]);
    __builtin_amdgcn_sched_barrier(0);
    load_k_sub<true>(a, lrow, j, q, 1, slot, kf[1]);
    // q fragments: tile u, column 8 (t % 2) + h = bf16(q) of row t = 2u + t % 2, head h, and + 4 its
    // low part (a missing row's columns stay as they are); wave w makes head w of every row
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int col = 8 * (t & 1) + wv;
        float o[4];
        if constexpr (PREP) {
            head_norm_rope_wave(a, a.proj + (size_t)(r0 + t) * kAttnInRows + (4 * j + wv) * 512, a.q_norm,
                                a.rm.pos[r0 + t], o);
        } else {
#pragma unroll
            for (int w = 0; w < 4; ++w) o[w] = a.q[((size_t)(r0 + t) * kNq + 4 * j + wv) * 256 + lane + 64 * w];
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint16_t hi = f2bf(o[w]);
            qbuf[t >> 1][col][lane + 64 * w] = hi;
            qbuf[t >> 1][col + 4][lane + 64 * w] = f2bf(o[w] - bf2f(hi));
        }
    }
    if (PREP && wv < T) {                               // row wv's new K / V row, if it is in this chunk
        const int sl = a.rm.slot[r0 + wv];
        if (sl / kChunk == c)
            make_kv_row(a, a.proj + (size_t)(r0 + wv) * kAttnInRows, a.rm.pos[r0 + wv], lrow, j, sl, knew[wv]);
    }
    __syncthreads();
    if (t0 > slot) return;
    q35_u32x4 qf[NU][8];
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int s = 0; s < 8; ++s) qf[u][s] = *(const q35_u32x4*)&qbuf[u][n][s * 32 + g * 8];
    const int tr = n >> 3;                               // this lane's row within a tile: 2u + tr
    int lslot[NU];                                       // that row's slot (-1: no such row)
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int ta = 2 * u, tb = 2 * u + 1 < T ? 2 * u + 1 : 2 * u;
        lslot[u] = tr == 0 ? slot_t[ta] : 2 * u + 1 < T ? slot_t[tb] : -1;
    }
    float(*ss)[4][kSegRow] = ss_all[wv];
    float sv[NU][4][4];
#pragma unroll
    for (int st = 0; st < 4; ++st) {
        if (PREP) {                                      // new K rows: their loads may be stale
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (slot_t[t] >> 4 == 4 * q + st && n == (slot_t[t] & 15)) {
#pragma unroll
                    for (int s = 0; s < 8; ++s) kf[st & 1][s] = *(const q35_u32x4*)&knew[t][s * 32 + g * 8];
                }
        }
        q35_f32x4 acc[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            acc[u] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; ++s)
                acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[st & 1][s], *(const q35_bf16x8*)&qf[u][s], acc[u], 0, 0, 0);
        }
        if (st < 2) load_k_sub<true>(a, lrow, j, q, st + 2, slot, kf[st & 1]);
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            q35_f32x4 scv;
            const int t = 2 * u + tr, tt0 = t0 + st * 16 + 4 * g;
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const float lo = row_down4(acc[u][rr]);   // lanes with n % 8 < 4 add the q_lo column
                const float sc = (acc[u][rr] + lo) * 0.0625f;
                const bool ok = (n & 7) < 4 && tt0 + rr <= lslot[u];
                sv[u][st][rr] = ok ? sc : -INFINITY;
                scv[rr] = sc;
            }
            if ((n & 7) < 4 && t < T) *(q35_f32x4*)&ss[t][n & 3][st * 16 + 4 * g] = scv;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        float m = -INFINITY;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) m = fmaxf(m, sv[u][st][rr]);
        m = fmaxf(m, xor16(m));
        m = fmaxf(m, xor32(m));
        float e = 0.f;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) e += sv[u][st][rr] > -INFINITY ? expf(sv[u][st][rr] - m) : 0.f;
        e += xor16(e);
        e += xor32(e);
        if (g == 0 && (n & 7) < 4 && 2 * u + tr < T) *(float2*)&ss[2 * u + tr][n & 3][64] = make_float2(m, e);
    }
    // a row's slice of scores as one contiguous KiB (slots past the row's last are never read), in
    // this form's own order of the scratch: [row][kv head][slice][head][64 slots]
    wave_sync();
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (t0 > slot_t[t]) continue;
        *(q35_f32x4*)(a.sc + (((size_t)(r0 + t) * kNkv + j) * (a.sc_ld / 64) + q) * 256 + lane * 4) =
            *(const q35_f32x4*)&ss[t][lane >> 4][(lane & 15) * 4];
        if (lane < 4)
            *(float2*)(a.stats + ((size_t)(r0 + t) * kNq + 4 * j + lane) * a.max_chunks * 8 + 2 * q) = *(const float2*)&ss[t][lane][64];
    }
}

// kSegParts x T x 4 KiB of dynamic LDS when a pair can have more than one segment
template <int T>
__global__ void __launch_bounds__(256, 2) attn_seg_pv(AttnArgs a, int nseg) {
    __shared__ uint16_t pl[16 * kPlStride];
    __shared__ float ml_all[T][4][2];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4;
    int pr, p0;
    if (!seg_of(a, nseg, pr, p0)) return;
    p0 *= kSegParts;
    const int j = pr % kNkv, r0 = (pr / kNkv) * T;
    int slot_t[T];
#pragma unroll
    for (int t = 0; t < T; ++t) slot_t[t] = a.rm.slot[r0 + t];
    int slot = slot_t[0];
#pragma unroll
    for (int t = 1; t < T; ++t) slot = max(slot, slot_t[t]);
    const int np = slot / kPart + 1, p1 = min(p0 + kSegParts, np);
    const int pown = (slot_t[0] + 1) / kPart;            // parts from pown on hold slots past the first row's
    if (p0 >= np) return;
    const int lrow = a.rm.lane[r0];
    const size_t sst = (size_t)a.max_chunks * 8;
    // the thread's two scores of a part per row (head idx / 128, slot idx % 128), loaded two parts
    // ahead and issued before that part's V (see attn_rows)
    auto load_scores = [&](int pc, float (&sr)[T][2]) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int idx = tid + q * 256, i = idx >> 7, tt = idx & 127;
                const int ts = min(pc * kPart + tt, slot);
                sr[t][q] = a.sc[(((size_t)(r0 + t) * kNkv + j) * (a.sc_ld / 64) + (ts >> 6)) * 256 + i * 64 + (ts & 63)];
            }
    };
    q35_u32x4 vfa[4][4], vfb[4][4];
    float sra[T][2], srb[T][2];
    load_scores(p0, sra);
    __builtin_amdgcn_sched_barrier(0);
    load_vf(a, lrow, j, p0, slot, 4 * wv, vfa);
    __builtin_amdgcn_sched_barrier(0);
    load_scores(p0 + 1, srb);
    __builtin_amdgcn_sched_barrier(0);
    load_vf(a, lrow, j, p0 + 1, slot, 4 * wv, vfb);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < T; ++t)
        softmax_ml(a.stats + ((size_t)(r0 + t) * kNq + 4 * j) * sst, sst, slot_t[t] / 64 + 1, ml_all[t]);
    const int myslot = g == 0 ? slot_t[0] : g == 1 ? slot_t[T > 1 ? 1 : 0] : slot_t[T > 2 ? 2 : 0];
    const bool whole = np <= kSegParts;                          // block-uniform: no other segment of this pair
    // the parts' sums wait in LDS, [P][T][4 waves][4 tiles][16 dims][4 heads], for the segment's end
    // (see attn_seg_scores)
    extern __shared__ __attribute__((aligned(16))) float seg_lds[];
    float* mypart = seg_lds + (min(g, T - 1) * 4 + wv) * 256 + (lane & 15) * 4;
    q35_f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
    auto part = [&](int pc, q35_u32x4 (&vf)[4][4], float (&sr)[T][2], auto more) {
        lds_barrier();          // ml is in; every wave is done with the previous part's weights
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int nn = min(kPart, slot_t[t] + 1 - pc * kPart);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int idx = tid + q * 256, i = idx >> 7, tt = idx & 127;
                pl[(4 * t + i) * kPlStride + tt] = tt < nn ? f2bf(expf(sr[t][q] - ml_all[t][i][0]) / ml_all[t][i][1]) : (uint16_t)0;
            }
        }
        lds_barrier();
        if (pc == np - 1) mask_vf(pc, slot, vf);
        q35_f32x4 out[4];
        pv_mfma(pl, 4 * T, vf, out);
        if (pc >= pown) pv_own_rows<T, 4>(pl, pc, slot_t, vf, out);
        if (decltype(more)::value) {
            load_scores(pc + 2, sr);
            load_vf(a, lrow, j, pc + 2, slot, 4 * wv, vf);
        }
        // lane (n, g) holds row g's four heads of dim 16 (4 wv + i) + n
        const bool mine = g < T && pc < myslot / kPart + 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!whole && g < T) *(q35_f32x4*)(mypart + (pc - p0) * T * 1024 + i * 64) = out[i];
            if (mine) acc[i] += out[i];
        }
    };
    int pc = p0;
    for (; pc + 2 < p1; pc += 2) {
        part(pc, vfa, sra, std::true_type{});
        part(pc + 1, vfb, srb, std::true_type{});
    }
    part(pc, vfa, sra, std::false_type{});
    if (pc + 1 < p1) part(pc + 1, vfb, srb, std::false_type{});
    if (!whole) {
        wave_sync();
        for (pc = p0; pc < p1; ++pc)
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (pc < slot_t[t] / kPart + 1)
                    *(q35_f32x4*)(a.part + part_offset(a, r0 + t, pc, j, 64 * wv) + lane * 4) =
                        *(const q35_f32x4*)(seg_lds + ((pc - p0) * T + t) * 1024 + wv * 256 + lane * 4);
        return;
    }
    if (g < T) store_gated<4>(a, r0 + g, j, 64 * wv + (lane & 15), acc);
}

// ---------------------------------------------------------------- prompt waves (flash form)
// A prompt wave of one lane (T >= 64 rows at consecutive slots): all of its rows read the
// same K/V, so a block takes 16 rows x the 4 q heads of one kv head (64 query columns) and
// streams the lane's K/V once for all of them, with both products on MFMA:
//   S^T = K Q^T   A = the K cache's fragments (16 slots x 32 dims per step), B = q as bf16 hi
//                 (8 steps) plus its lo part on the rotated dims 0..63 (2 steps): the
//                 decode path's split of the f32 post-rope q; wave w owns columns
//                 (row 4w + n/4, head n%4) and streams every K tile itself
//   online softmax per column over 64-slot tiles (running max and sum in f32, e^(s - m)
//                 rounded to bf16 as the P.V operand)
//   O = P V       A = P straight from the S^T accumulators (lane (column, g) holds slots
//                 4g + r of each 16-slot sub-tile: the MFMA's k index is taken in that order),
//                 B = V from LDS, staged by all 4 waves in the cache's 8-slot layout, where a
//                 lane's 4 slots of one dim are one 8-byte read
// The softmax normalisation comes last (O / l), so the bf16 rounding of the weights happens
// before it rather than after as on the decode path (speccheck/specimpl.py:385-392 rounds
// the normalised weights): same math, different rounding point -- prompt logits stay within
// the engine-vs-oracle tolerance, not bit-equal to the one-row kernels.
constexpr int kPrRows = 16;
typedef short q35_s16x4 __attribute__((ext_vector_type(4)));

// V tile in LDS: the cache's 8-slot layout (kv_v8_offset) as it stands, 8 groups x 256 dims x
// 8 slots (32 KiB); a lane's 4 slots of one dim are one 8-byte read, every read address one
// lane base plus an immediate offset
constexpr int kPrVBuf = 64 * 256 * 2;                       // bytes per V tile


constexpr int kPrLds = 2 * 64 * 256 * 2 + 2 * kPrVBuf;   // K and V tiles, double-buffered: 128 KiB

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 q35_bf16x2;
// two f32 -> packed bf16 (round to nearest even, v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
    const q35_bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

__global__ void __launch_bounds__(256) attn_prompt(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t pr_lds[];
    uint16_t(*kt)[64 * 256] = (uint16_t(*)[64 * 256])pr_lds;
    uint16_t* vt = pr_lds + 2 * 64 * 256;                          // [2][8 groups][256 dims][8 slots]
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int T = a.T, ngrp = (T + kPrRows - 1) / kPrRows;
    // XCDs 0-3 take kv head 0 and 4-7 kv head 1: each XCD's L2 holds one head's K/V stream
    const int xcd = blockIdx.x & 7, j = xcd >> 2;
    const int grp = (blockIdx.x >> 3) * 4 + (xcd & 3);
    if (grp >= ngrp) return;
    const int r0 = grp * kPrRows;
    const int lrow = a.rm.lane[0];
    const int smax = a.rm.slot[min(r0 + kPrRows, T) - 1];
    const int qrow = min(r0 + 4 * wv + (n >> 2), T - 1);
    const int qslot = a.rm.slot[qrow];
    const int wslot = a.rm.slot[min(r0 + 4 * wv, T - 1)];     // the wave's smallest slot
    const size_t kvbase = lrow * a.kv_lane + a.kv_layer_off + (size_t)j * a.cap * 256;

    // q fragments of column n: dims s*32 + g*8 .. +8
    q35_u32x4 qhi[8], qlo[2];
    {
        const float* qp = a.q + ((size_t)qrow * kNq + 4 * j + (n & 3)) * 256 + g * 8;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const float4 x0 = *(const float4*)(qp + s * 32), x1 = *(const float4*)(qp + s * 32 + 4);
            const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            uint16_t h[8], l[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                h[e] = f2bf(xs[e]);
                l[e] = f2bf(xs[e] - bf2f(h[e]));
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) qhi[s][e] = (uint32_t)h[2 * e] | ((uint32_t)h[2 * e + 1] << 16);
            if (s < 2) {
#pragma unroll
                for (int e = 0; e < 4; ++e) qlo[s][e] = (uint32_t)l[2 * e] | ((uint32_t)l[2 * e + 1] << 16);
            }
        }
    }
    const int ntiles = smax / 64 + 1;
    // K and V tiles (64 slots) reach LDS by direct-to-LDS loads (global_load_lds: lane i of
    // an instruction fills the 16-byte slot i of a 1 KiB run), issued one tile ahead: K in its
    // cache layout (four 16-slot MFMA tiles, 32 KiB contiguous), V in its 8-slot layout (eight
    // 4 KiB groups, contiguous). Cached loads: the 12 blocks of a kv head on one XCD read
    // the same tiles and all but the first hit that XCD's L2. Tiles and groups past the group's
    // last slot are clamped to it (K: scores masked; V: weights zero, and the values of slots
    // past the last are zeroed where they are read, in the last tile). The wave's 8 K and 8 V
    // runs per tile are its only vector-memory loads in the loop, so "s_waitcnt vmcnt(0)"
    // at the top of a tile waits for exactly that tile's data; every LDS read below is
    // inline asm, which keeps the compiler from waiting on the prefetch in flight.
    auto issue_tiles = [&](int it, int buf) {
        const int t0 = it * 64;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int run = wv * 8 + i;                   // 1 KiB run of the 32 KiB tile
            const int tile = min(it * 4 + (run >> 3), smax >> 4);
            __builtin_amdgcn_global_load_lds(
                (const void*)(a.kc + kvbase + (size_t)tile * 4096 + (run & 7) * 512 + lane * 8),
                (__attribute__((address_space(3))) void*)&kt[buf][run * 512], 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int run = wv * 8 + i;                   // 1 KiB run: group run / 4, dims 64 (run % 4) ..
            const int grp = min(t0 / 8 + (run >> 2), smax >> 3);
            __builtin_amdgcn_global_load_lds(
                (const void*)(a.vc + kvbase + (size_t)grp * 2048 + (run & 3) * 512 + lane * 8),
                (__attribute__((address_space(3))) void*)(vt + buf * (kPrVBuf / 2) + run * 512), 16, 0, 0);
        }
    };
    issue_tiles(0, 0);

    float m_run = -INFINITY, l_run = 0.f;
    q35_f32x4 o[16];
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) o[dt] = (q35_f32x4){0.f, 0.f, 0.f, 0.f};
    // LDS byte offsets: K fragment (sub-tile st, step s) at st*8192 + s*1024 + lane*16; V:
    // lane (n, g) reads slots 32ks + 16c + 4g .. +4 of dim 16 dt + n, i.e. group 4ks + 2c + g/2,
    // slots 4 (g % 2) .. +4: the lane's base plus the immediate (4ks + 2c) * 4096 + 256 dt
    const unsigned kb0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)&kt[0][0] + lane * 16;
    const unsigned vlane = (unsigned)(size_t)(__attribute__((address_space(3))) void*)vt +
                           (unsigned)(((g >> 1) * 2048 + n * 8 + 4 * (g & 1)) * 2);

    for (int it = 0; it < ntiles; ++it) {
        const int t0 = it * 64, buf = it & 1;
        // this tile's loads have landed (the only ones in flight), and every wave is done
        // with the other buffer (tile it - 1) before it is refilled
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (it + 1 < ntiles) issue_tiles(it + 1, buf ^ 1);
        const unsigned kbase = kb0 + (unsigned)(buf * 64 * 256 * 2);
        float sv[4][4];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            q35_u32x4 kf[8];
#pragma unroll
            for (int s = 0; s < 8; ++s)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[s]) : "v"(kbase), "n"(st * 8192 + s * 1024) : "memory");
            asm volatile("s_waitcnt lgkmcnt(0)"
                         : "+v"(kf[0]), "+v"(kf[1]), "+v"(kf[2]), "+v"(kf[3]), "+v"(kf[4]), "+v"(kf[5]), "+v"(kf[6]), "+v"(kf[7]));
            q35_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; ++s)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[s], *(q35_bf16x8*)&qhi[s], acc, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&kf[s], *(q35_bf16x8*)&qlo[s], acc, 0, 0, 0);
            // scores in the log2 domain: s / 16 * log2(e)
#pragma unroll
            for (int r = 0; r < 4; ++r) sv[st][r] = acc[r] * (0.0625f * 1.4426950408889634f);
        }
        if (t0 + 63 > wslot) {            // a tile crossing the diagonal of some column of the wave
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (t0 + st * 16 + 4 * g + r > qslot) sv[st][r] = -INFINITY;
        }
        // online softmax of column n over this tile
        float mt = -INFINITY;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int r = 0; r < 4; ++r) mt = fmaxf(mt, sv[st][r]);
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, xor32(mt));
        const float mnew = fmaxf(m_run, mt);      // finite: slot 0 is in every column's first tile
        const float alpha = __builtin_amdgcn_exp2f(m_run - mnew);   // exp2(-inf) = 0 on the first tile
        // P as the A operand, bf16 (k = g*8 + e <-> slot 32 ks + 16 (e / 4) + 4g + e % 4); the
        // running sum adds the rounded weights that P.V uses
        q35_u32x4 pa[2];
        float ps = 0.f;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            float pv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) pv[r] = __builtin_amdgcn_exp2f(sv[st][r] - mnew);   // masked: 0
            const uint32_t w0 = pk_bf16(pv[0], pv[1]), w1 = pk_bf16(pv[2], pv[3]);
            pa[st >> 1][2 * (st & 1)] = w0;
            pa[st >> 1][2 * (st & 1) + 1] = w1;
            ps += (__uint_as_float(w0 << 16) + __uint_as_float(w0 & 0xffff0000u)) +
                  (__uint_as_float(w1 << 16) + __uint_as_float(w1 & 0xffff0000u));
        }
        ps += __shfl_xor(ps, 16, 64);
        ps += xor32(ps);
        l_run = l_run * alpha + ps;
        m_run = mnew;
        // rescale O rows 4g + r by their columns' alpha -- only when some column's max moved
        if (__any(alpha != 1.f)) {
            float ar[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
            for (int dt = 0; dt < 16; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[dt][r] *= ar[r];
        }
        // P.V: V fragments 8 d-tiles at a time (16 reads, one wait, 8 MFMAs); in the last tile
        // the values of slots past the group's last are zeroed (their memory is not initialised)
        const unsigned vb = vlane + (unsigned)(buf * kPrVBuf);
        const bool last = it == ntiles - 1;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            uint2 mk[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int cnt = last ? smax + 1 - (t0 + 32 * ks + 16 * c + 4 * g) : 4;   // valid slots of the 4
                mk[c] = (uint2){(cnt > 0 ? 0xffffu : 0u) | (cnt > 1 ? 0xffff0000u : 0u),
                                (cnt > 2 ? 0xffffu : 0u) | (cnt > 3 ? 0xffff0000u : 0u)};
            }
#pragma unroll
            for (int dh = 0; dh < 2; ++dh) {
                uint2 v0[8], v1[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v0[u])
                                 : "v"(vb), "n"((4 * ks) * 4096 + 256 * (8 * dh + u)) : "memory");
                    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v1[u])
                                 : "v"(vb), "n"((4 * ks + 2) * 4096 + 256 * (8 * dh + u)) : "memory");
                }
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(v0[0]), "+v"(v0[1]), "+v"(v0[2]), "+v"(v0[3]), "+v"(v0[4]), "+v"(v0[5]), "+v"(v0[6]), "+v"(v0[7]),
                               "+v"(v1[0]), "+v"(v1[1]), "+v"(v1[2]), "+v"(v1[3]), "+v"(v1[4]), "+v"(v1[5]), "+v"(v1[6]), "+v"(v1[7]));
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    q35_u32x4 b = {v0[u].x & mk[0].x, v0[u].y & mk[0].y, v1[u].x & mk[1].x, v1[u].y & mk[1].y};
                    o[8 * dh + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(q35_bf16x8*)&pa[ks], *(q35_bf16x8*)&b,
                                                                           o[8 * dh + u], 0, 0, 0);
                }
            }
        }
    }
    // O / l, bf16, times bf16(sigmoid(gate)): lane (n, g) holds row 4 wv + g, head r, dims 16 dt + n
    const int row = r0 + 4 * wv + g;
    float lr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) lr[r] = __shfl(l_run, 4 * g + r, 64);
    if (row < T) {
        // every gate value loaded before the first store (a store to out could alias proj,
        // which would otherwise serialize each load behind the previous store)
        const uint16_t* pr = a.proj + (size_t)row * kAttnInRows + 256 + n;
        uint16_t gv[4][16];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int dt = 0; dt < 16; ++dt) gv[r][dt] = pr[(4 * j + r) * 512 + 16 * dt];
        uint16_t* po = a.out + (size_t)row * 2048 + 4 * j * 256 + n;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int dt = 0; dt < 16; ++dt) {
                const float ov = rbf(o[dt][r] / lr[r]);
                const float gt = rbf(sigmoid_f(bf2f(gv[r][dt])));
                const int col = (4 * j + r) * 256 + 16 * dt + n;
                if (a.out_tiled) a.out[tiled_offset(row, col, 2048)] = f2bf(ov * gt);
                else po[r * 256 + 16 * dt] = f2bf(ov * gt);
            }
        }
    }
}

hipError_t attn_init() {
    const struct { const void* f; int lds; } big[] = {
        {(const void*)attn_fused<true, 1, true>, 96 * 1024}, {(const void*)attn_fused<true, 1, false>, 96 * 1024},
        {(const void*)attn_fused<false, 1, false>, 96 * 1024},
        {(const void*)attn_fused<true, 2, true>, kFused2MaxLds}, {(const void*)attn_fused<true, 2, false>, kFused2MaxLds},
        {(const void*)attn_rows<2, 8, true>, kRowsLdsDyn8}, {(const void*)attn_rows<2, 8, false>, kRowsLdsDyn8},
        {(const void*)attn_rows<3, 8, true>, kRowsLdsDyn8}, {(const void*)attn_rows<3, 8, false>, kRowsLdsDyn8}};
    for (const auto& b : big) {
        const hipError_t e = hipFuncSetAttribute(b.f, hipFuncAttributeMaxDynamicSharedMemorySize, b.lds);
        if (e != hipSuccess) return e;
    }
    return hipFuncSetAttribute((const void*)attn_prompt, hipFuncAttributeMaxDynamicSharedMemorySize, kPrLds);
}

static size_t fused_lds(const AttnArgs& a) {
    return (size_t)(4 * ((a.cap + 63) / 64 * 64) + 4 * 8 * a.max_chunks) * 4;
}
static bool fused_fits(const AttnArgs& a) { return fused_lds(a) <= 96 * 1024; }
static bool use_fused(const AttnArgs& a) {
    if (a.force == kAttnFused || a.force == kAttnFusedPair) return fused_fits(a);
    if (a.force != kAttnAuto) return false;
    return a.R >= 64 && fused_fits(a);
}
// Two items per block (one row per lane) when both items' LDS fits the CU and there are more items
// than CUs: up to 256 of them run one per CU, where pairing would leave half of the CUs idle and
// let the longer lane of a pair hold up the shorter one. us, one item -> two per block: 64 lanes x
// 4,000 slots 127 -> 193, 128 x 1,000 67 -> 76, 128 x 500 .. 4,000 ragged 137 -> 192; beyond, 160 x
// 4,000 263 -> 231, 160 x 1,000 88 -> 81. (Below 64 lanes the split path: 48 x 4,000 103, one item
// per block 127; 48 x 1,000 49 and 55.)
static bool use_fused2(const AttnArgs& a) {
    if (a.force == kAttnFused || a.T != 1 || 2 * fused_lds(a) > (size_t)kFused2MaxLds) return false;
    return a.force == kAttnFusedPair || (a.fused_pair && a.R * kNkv > 256);
}
// A lane's 2-3 verify rows in one block from 192 rows on: the K/V stream once instead of once per
// row. us, one block per row -> rows form: 100 lanes x 2 x 3,000 171 -> 123, ragged 143 -> 101; 64 x 3
// x 4,000 185 -> 145, ragged 138 -> 125; 64 x 3 x 1,000 58.6 -> 59.3, 64 x 2 x 4,000 125 -> 127, 32 x 3 x
// 4,000 99 -> 124. A block streams its lane's slots at 22.5 ns each, the full chip all lanes' at 0.45, so
// with less than 40 of the longest lane's slots in all the longest lane alone sets the time, and the
// segments cut it up. us, rows form -> segments: 64 x 3, 1 lane of 4,096 and the others of 128 120 -> 62,
// of 32,768 and 1,000 741 -> 139; a third of 80 lanes of 4,000, the others of 500 (33 times) 126 -> 112; 64
// lanes of 512 .. 4,096 (36) 126 -> 118, 80 (45) 131 -> 134; below 3,000 slots the two more launches
// weigh more: 64 of 250 .. 2,000 78 -> 82.
static int rows_w(const AttnArgs& a) { return a.rows_form == 2 ? 8 : 4; }
static bool uneven(const AttnArgs& a) { return a.ctx_max >= 3000 && a.ctx_sum < 40ll * a.ctx_max; }
static bool use_rows(const AttnArgs& a) {
    // the slice stats (and the tail) fit the block's dynamic LDS
    const bool shape = (a.T == 2 || a.T == 3) && a.R % a.T == 0 &&
                       rows_lds_bytes(a.T, a.max_chunks, rows_w(a)) <= (rows_w(a) == 8 ? (size_t)kRowsLdsDyn8 : 65536);
    if (a.force == kAttnRows) return shape;
    if (a.force != kAttnAuto) return false;
    return a.rows_form && shape && a.R >= 192 && !uneven(a);
}
// Verify rows by segments where the rows form is not taken and there are slots enough for two more
// launches; by the lanes' contexts, not their capacity, which may be mostly empty. us, all with another
// layer's K/V from call to call. Split path -> segments, three rows: 3 lanes x 8,192 slots 62 -> 52, 5 x
// 4,096 57 -> 48, 8 x 2,000 47 -> 48, 8 x 500 35 -> 43, 3 x 4,096 46 -> 47, 16 x 1,000 48 -> 49, 31 x 500 53 -> 45,
// 24 x 8,192 297 -> 125. Two rows (the split path reads the K/V only twice then): 16 x 3,000 62 -> 62, 16 x
// 4,000 74 -> 65, 22 x 4,000 ragged 65 -> 68, 31 x 2,000 78 -> 66, 31 x 1,000 56 -> 59, 48 x 500 51 -> 53, 80 x 500
// 65 -> 60. One lane's P.V segments are few blocks and its parts' sum is as long as the split path's:
// 500 slots 33 -> 42, 32,768 84 -> 86, 65,536 154 -> 160. Fused form, a block per row, -> segments: 31 lanes x
// 3 rows x 1,000 50 -> 55, 1,500 59 -> 61, 2,000 69 -> 64, 4,000 106 -> 91; 32 x 2 x 2,000 70 -> 66, 40 x 2 x 2,000
// 74 -> 77, 2,500 84 -> 81.
static bool use_seg(const AttnArgs& a) {
    if (a.force != kAttnAuto || (a.T != 2 && a.T != 3) || a.R % a.T || a.R == a.T || use_rows(a)) return false;
    if (a.R >= 192 && uneven(a)) return true;
    if (use_fused(a)) return a.R < 96 && a.ctx_max >= (a.T == 2 ? 2048 : 1536);
    return a.T == 2 ? a.ctx_sum + 200ll * a.R >= 54000 : a.ctx_sum + 150ll * a.R >= 18000;
}
static bool use_prompt(const AttnArgs& a) {
    const bool shape = a.T >= 64 && a.R == a.T;
    if (a.force == kAttnPrompt) return shape;
    if (a.force != kAttnAuto) return false;
    return a.prompt_flash && shape;
}

// The form makes q and the new K / V rows itself: the split and the fused form with one row per lane, the
// rows form and the segments, whose blocks read only rows they make, as long as no lane occurs twice
// (another row's block would append to the lane while this one reads it). The fused form up to
// 600,000 slots in all: there the launch it saves is 2 .. 8 % (us, attn_prep -> folded: 256 lanes x
// 1,000 slots 117.4 -> 113.9, 130 x 4,000 223 -> 212); beyond it a full chip streaming at the HBM
// rate pays more for every block's appended rows at once (224 x 3,000 237 -> 242, 240 x 4,000 323
// -> 350). The rows form gains everywhere (250 lanes x 3 rows x 2,000: 200 -> 198, ragged 158 -> 151).
static bool prep_folded(const AttnArgs& a) {
    if (use_prompt(a) || !a.distinct) return false;
    if (use_rows(a) || use_seg(a)) return true;
    return a.T == 1 && (!use_fused(a) || (long long)a.R * a.cap <= 600000);
}

bool attn_prompt_form(const AttnArgs& a) { return use_prompt(a); }

// Whether the forced form can run this shape (kAttnAuto always can).
bool attn_form_ok(const AttnArgs& a) {
    switch (a.force) {
    case kAttnAuto: case kAttnSplit: case kAttnSplit4: return true;
    case kAttnFused: return use_fused(a) && a.R % a.T == 0;
    case kAttnFusedPair: return use_fused(a) && use_fused2(a);
    case kAttnRows: return use_rows(a);
    case kAttnPrompt: return use_prompt(a);
    default: return false;
    }
}

hipError_t launch_attn_prep(const AttnArgs& a, hipStream_t st) {
    if (a.R <= 0 || a.max_chunks <= 0) return hipErrorInvalidValue;
    if (prep_folded(a)) return hipSuccess;
    hipLaunchKernelGGL(attn_prep, dim3((a.R * (kNq + kNkv) + 3) / 4), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_attn_core(const AttnArgs& a, hipStream_t st) {
    if (a.R <= 0 || a.max_chunks <= 0) return hipErrorInvalidValue;
    if (a.T > 1 && (a.ctx_max <= 0 || a.ctx_max > a.cap)) return hipErrorInvalidValue;
    const int lds_slots = (a.cap + 63) / 64 * 64;
    const size_t lds = fused_lds(a);
    if (!attn_form_ok(a)) return hipErrorInvalidValue;
    if (use_prompt(a)) {
        // one lane's prompt wave: 16 rows per block, kv head by XCD half
        const int ngrp = (a.T + kPrRows - 1) / kPrRows;
        hipLaunchKernelGGL(attn_prompt, dim3((ngrp + 3) / 4 * 8), dim3(256), kPrLds, st, a);
    } else if (use_rows(a)) {
        const int W = rows_w(a);
        const size_t lds = rows_lds_bytes(a.T, a.max_chunks, W);
#define Q35_ROWS(TV, WV)                                                                                          \
    if (a.T == TV && W == WV) {                                                                                   \
        if (prep_folded(a)) hipLaunchKernelGGL((attn_rows<TV, WV, true>), dim3(a.R / TV * kNkv), dim3(64 * WV), lds, st, a); \
        else hipLaunchKernelGGL((attn_rows<TV, WV, false>), dim3(a.R / TV * kNkv), dim3(64 * WV), lds, st, a);     \
    }
        Q35_ROWS(2, 8) Q35_ROWS(3, 8) Q35_ROWS(2, 4) Q35_ROWS(3, 4)
#undef Q35_ROWS
    } else if (use_seg(a)) {
        // blocks up to the longest lane's last slot
        const int pairs = (a.R / a.T * kNkv + 7) / 8 * 8, ns = (a.ctx_max + kChunk - 1) / kChunk;
        const int np = (a.ctx_max + kPart * kSegParts - 1) / (kPart * kSegParts);
        const size_t lp = np > 1 ? (size_t)kSegParts * a.T * 4096 : 0;
#define Q35_SEG(TV)                                                                                              \
    if (a.T == TV) {                                                                                             \
        if (prep_folded(a)) hipLaunchKernelGGL((attn_seg_scores<TV, true>), dim3(pairs * ns), dim3(256), 0, st, a, ns); \
        else hipLaunchKernelGGL((attn_seg_scores<TV, false>), dim3(pairs * ns), dim3(256), 0, st, a, ns);        \
        hipLaunchKernelGGL((attn_seg_pv<TV>), dim3(pairs * np), dim3(256), lp, st, a, np);                       \
    }
        Q35_SEG(2) Q35_SEG(3)
#undef Q35_SEG
        if (np > 1) hipLaunchKernelGGL(attn_combine, dim3(a.R, kNq), dim3(256), 0, st, a, kSegParts);
    } else if (use_fused(a)) {
        if (a.T < 1 || a.R % a.T) return hipErrorInvalidValue;
        const int pairs = a.R / a.T * kNkv;
        const int nseg = std::max(1, 8 / pairs), seg = (a.T + nseg - 1) / nseg;
        const dim3 grid((pairs * nseg + 7) / 8 * seg * 8);
        const bool prep = prep_folded(a);
        if (use_fused2(a)) {
            const dim3 g2((grid.x + 15) / 16 * 8);
            if (prep) hipLaunchKernelGGL((attn_fused<true, 2, true>), g2, dim3(512), 2 * lds, st, a, lds_slots);
            else hipLaunchKernelGGL((attn_fused<true, 2, false>), g2, dim3(512), 2 * lds, st, a, lds_slots);
        } else if (a.T == 1) {
            if (prep) hipLaunchKernelGGL((attn_fused<true, 1, true>), grid, dim3(256), lds, st, a, lds_slots);
            else hipLaunchKernelGGL((attn_fused<true, 1, false>), grid, dim3(256), lds, st, a, lds_slots);
        } else {
            hipLaunchKernelGGL((attn_fused<false, 1, false>), grid, dim3(256), lds, st, a, lds_slots);
        }
    } else {
        // chunks that can hold a row's slots (with one row per lane all of the capacity's: a captured step's
        // positions move on)
        const int nc = a.T > 1 ? (a.ctx_max + kChunk - 1) / kChunk : a.max_chunks;
        if (a.force == kAttnSplit4 || (a.force != kAttnSplit && a.split4)) {
            if (prep_folded(a))
                hipLaunchKernelGGL(attn_scores4<true>, dim3(a.R, kNkv, nc * 4), dim3(256), 0, st, a);
            else
                hipLaunchKernelGGL(attn_scores4<false>, dim3(a.R, kNkv, nc * 4), dim3(256), 0, st, a);
            hipLaunchKernelGGL(attn_pv4, dim3(a.R, kNkv, nc * 8), dim3(64), 0, st, a);
        } else {
            if (prep_folded(a))
                hipLaunchKernelGGL(attn_scores_prep, dim3(a.R, kNkv, nc * 4), dim3(64), 0, st, a);
            else
                hipLaunchKernelGGL(attn_scores, dim3(a.R, kNkv, nc * 4), dim3(64), 0, st, a);
            hipLaunchKernelGGL(attn_pv, dim3(a.R, kNkv, nc * 2), dim3(256), 0, st, a);
        }
        hipLaunchKernelGGL(attn_combine, dim3(a.R, kNq), dim3(256), 0, st, a, 0);
    }
    return hipGetLastError();
}

}  // namespace q35
