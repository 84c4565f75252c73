// GQA flash-decode for gfx950 over short contexts: one new position per sequence, f16 KV, head_dim 128, no split of the
// context and no merge launch.
//
// A compute unit reads 57 GB/s from HBM however its wavefronts ask for it, 16 KB of keys and values (a 32-key block) in
// 0.28 us, so a step whose contexts stay whole lasts as long as the longest of them; cutting the context instead
// costs a merge launch, 2.4 us and more. Here a (slot, KV head) is cut by channels: each of P workgroups works
// out all scores, from all the keys, and the output of its own 128 / P channels, from that part of the values. A block is
// 8 + 8 / P KB to a compute unit, and nothing is left to merge but the workgroup's own wavefronts.
//   - eight wavefronts, R = 1 to 3 blocks each, every load asked for before the first is waited for: no loop, one maximum
//     over a wavefront's blocks, nothing rescaled;
//   - S^T = K . Q^T and O^T = V^T . P^T as in attn_decode_f16.hip; the scale goes to the scores, as there, or to the queries
//     on their way to f16, as in the split-K kernel: to what it goes in the form that the step has where it may not go by
//     channels, so that channels which fit f16 only with the scale on, or only without it, fit in either;
//   - wavefront 0 of every workgroup converts the new position's row, the wavefront that has its block patches it into its
//     operands, and the first part's workgroup stores it.
// The parts of up to eight KV heads follow one another that many workgroups apart: workgroup i runs on compute die
// i mod 8, so with eight heads the parts of one find its keys in one L2.
// 32 Q / 4 KV heads, us a layer, the split-K kernel's whole and split steps before -> this: one slot at 83 / 200 / 300 / 370 /
// 500 positions 3.9 / 5.9 / 6.7 / 7.2 / 6.2 -> 3.5 / 3.9 / 4.8 / 4.9 / 5.2 (8 parts), 16 slots at 83 / 200 / 300 / 500 / 700
// 5.1 / 7.2 / 8.1 / 9.9 / 11.8 -> 4.8 / 5.4 / 6.2 / 7.6 / 9.3 (4 parts), preparing, one slot at 0 / 200 / 300
// 4.9 / 6.8 / 7.3 -> 4.1 / 4.4 / 5.3. What bounds it now: 2.4 us of launch and first trips to memory, then the compute unit's
// 9 KB a block. In place of blocks beyond the last, loads that read as much as the others cost 1 us at 17 blocks
// (slots=4 7.1 against 6.6), so those read one line each.
//
// Semantics: as attn_decode_f16.hip.
#include "internal.h"
#include "mfma_common.h"
#include "prep_fold.h"
#include "split_exchange.h"

#include <math.h>

#include <algorithm>

namespace itak {

namespace {

constexpr int kWaves = 8;

__device__ __forceinline__ float column_max4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float column_sum4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// P parts; R blocks a wavefront. PREP: Q and the new K row are normed and rotated on their way in (prep_fold.h) and
// the gate is applied to the output.
template <int N, bool RING, bool PREP, int P, int R>
__device__ __forceinline__ void attn_whole_f16_body(const AttnParams &p, const AttnBatchT<N> &b,
                                                    [[maybe_unused]] const FoldedParams &fold) {
    constexpr int kT = 8 / P;  // channel tiles of a part
    __shared__ float sm_m[kWaves * 16], sm_l[kWaves * 16];
    __shared__ __attribute__((aligned(16))) float sm_o[kWaves * kT * 256];
    __shared__ __attribute__((aligned(16))) _Float16 sm_q[16 * kQStride];
    __shared__ __attribute__((aligned(16))) _Float16 sm_new[2 * kD];  // the new K row, then the new V row

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t g = lane >> 4, jl = lane & 15;
    // (Every kernel argument in one batch of scalar loads.)
    if (N == 1)
        asm volatile("" ::"s"(p.layer_base), "s"(p.q), "s"(p.out), "s"(p.k_new), "s"(p.v_new), "s"(p.g.slot_stride),
                     "s"(p.g.head_stride), "s"(p.g.side_stride), "s"(p.g.kv_heads), "s"(p.q_heads), "s"(p.group), "s"(p.scale),
                     "s"(p.softcap), "s"(p.scale_scores), "s"(b.item[0].slot), "s"(b.item[0].q_row0), "s"(b.item[0].kv_len),
                     "s"(b.item[0].kv_lo), "s"(p.window), "s"(p.ring_blocks));
    if (N == 1 && PREP)
        asm volatile("" ::"s"(fold.prep_q_weight), "s"(fold.prep_k_weight), "s"(fold.prep_eps), "s"(fold.prep_rot),
                     "s"(fold.prep_interleaved), "s"(fold.prep_freq_step), "s"(fold.prep_freq), "s"(fold.gate));
    const AttnItem item = b.of_block(blockIdx.x);
    const uint32_t local = blockIdx.x - item.block0, heads = p.g.kv_heads, group = p.group;
    const uint32_t eight = local / (8 * P), in = local - eight * 8 * P, held = min(8u, heads - eight * 8);
    uint32_t part = 0;
#pragma unroll
    for (int x = 1; x < P; ++x) part += in >= x * held ? 1u : 0u;
    const uint32_t kv_head = eight * 8 + in - part * held;

    uint16_t *kplane = static_cast<uint16_t *>(const_cast<void *>(p.layer_base)) + item.slot * p.g.slot_stride +
                       kv_head * p.g.head_stride;
    uint16_t *vplane = kplane + p.g.side_stride;
    const uint32_t pos = item.kv_len - 1;  // the query's position: the newest row
    const uint32_t kb_begin = RING ? item_first_block(item) : 0, kb_end = (item.kv_len + kBlockKeys - 1) / kBlockKeys;
    const uint32_t ring_blocks = RING ? p.ring_blocks : 0;

    // ---- every load. Queries first: thread f holds channels 4*(f%32) .. +3 of vector f/32; vectors beyond the
    // group re-read the last real one and are zeroed when staged.
    const uint32_t qj = tid >> 5, c4 = (tid & 31) * 4;
    float4 qraw = *reinterpret_cast<const float4 *>(
        p.q + (uint64_t(item.q_row0) * p.q_heads + kv_head * group + min(qj, group - 1)) * kD + c4);
    // The new row: lanes 0..31 of wavefront 0 the keys', 32..63 the values'.
    const bool fused = p.k_new != nullptr;
    float4 nraw = make_float4(0.f, 0.f, 0.f, 0.f);
    if (fused && wave == 0)
        nraw = *reinterpret_cast<const float4 *>((lane < 32 ? p.k_new : p.v_new) +
                                                 (uint64_t(item.q_row0) * heads + kv_head) * kD + c4);
    // PREP: the norm weights and the frequencies of this lane's four channels.
    const uint32_t prot = PREP ? fold.prep_rot : 0;
    const bool pinter = PREP && fold.prep_interleaved != 0;
    const int trig_pairs = pinter ? 2 : 4;
    [[maybe_unused]] const uint32_t pair0 = pinter ? c4 >> 1 : (c4 < prot >> 1 ? c4 : c4 - (prot >> 1));
    [[maybe_unused]] float4 wq = make_float4(1.f, 1.f, 1.f, 1.f), wk = wq;
    [[maybe_unused]] double freq[4] = {0.0, 0.0, 0.0, 0.0};
    if constexpr (PREP) {
        if (fold.prep_q_weight) wq = *reinterpret_cast<const float4 *>(fold.prep_q_weight + c4);
        if (fold.prep_k_weight) wk = *reinterpret_cast<const float4 *>(fold.prep_k_weight + c4);
        if (prot && fold.prep_freq) {
#pragma unroll
            for (int i = 0; i < 4; ++i) freq[i] = fold.prep_freq[min(pair0 + i, (prot >> 1) - 1)];
        }
    }
    // The wavefront's blocks: wave, wave + 8, .. from the first. In place of one beyond the last every lane loads the same 16 bytes
    // of the first, one line a load: a branch round the loads would have every wait behind it wait for all of them.
    half8 bk[R][2][4], bv[R][kT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves;
        const bool has = kb < kb_end;
        uint32_t sb = has ? kb : kb_begin;
        if (RING) sb %= ring_blocks;
        const uint16_t *base = kplane + uint64_t(sb) * (kBlockKeys * kD) + (has ? (g * 16 + jl) * 8 : 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                bk[r][t][s] = *reinterpret_cast<const half8 *>(base + ((t * 16 + s * 4) * 16) * 8);
        __builtin_amdgcn_sched_barrier(0);  // (in their order: the first block's products wait for the first loads alone)
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves;
        const bool has = kb < kb_end;
        uint32_t sb = has ? kb : kb_begin;
        if (RING) sb %= ring_blocks;
        const uint16_t *base = vplane + uint64_t(sb) * (kBlockKeys * kD) + part * kT * 16 * kBlockKeys + (has ? jl * kBlockKeys + g * 8 : 0);
#pragma unroll
        for (int c = 0; c < kT; ++c)
            bv[r][c] = __builtin_nontemporal_load(reinterpret_cast<const half8 *>(base + c * 16 * kBlockKeys));
    }
    // What this thread finishes: value tid + 512 u of the part's outputs, [tile][lane][register] as the wavefronts leave them.
    constexpr int kF = P == 8 ? 1 : kT * 256 / (kWaves * 64);  // (of eight parts half the threads do)
    const uint32_t fcol = (tid >> 2) & 15, fch = part * kT * 16 + (P == 8 ? 0 : tid >> 8) * 16 + ((tid >> 6) & 3) * 4 + (tid & 3);
    const uint64_t out_at = (uint64_t(item.q_row0) * p.q_heads + kv_head * group + min(fcol, group - 1)) * kD + fch;
    [[maybe_unused]] float gt[kF];
    if constexpr (PREP) {
#pragma unroll
        for (int u = 0; u < kF; ++u) gt[u] = (fold.gate ? fold.gate : p.q)[out_at + u * 32];
    }

    const float softcap = p.softcap;
    const float scale = softcap > 0.0f ? p.scale : p.scale * kLog2e;
    // The queries are rounded to f16 with the scale on, or as they are and the scale goes to the scores, as the planner says.
    const bool scale_scores = !PREP && p.scale_scores != 0;
    const float qscale = scale_scores ? 1.0f : scale, score_scale = scale_scores ? scale : 1.0f;
    [[maybe_unused]] PrepTrig trig;
    if constexpr (PREP) {
        if (prot) {
            if (!fold.prep_freq)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i < trig_pairs) freq[i] = exp2(double(pair0 + i) * fold.prep_freq_step);
            prep_trig(trig, double(pos), freq, trig_pairs);
        }
        qraw = prep_chunk(qraw, fold.prep_q_weight != nullptr, wq, fold.prep_eps, c4, lane, prot, pinter, trig);
    }
    {
        half4 h{static_cast<_Float16>(qraw.x * qscale), static_cast<_Float16>(qraw.y * qscale),
                static_cast<_Float16>(qraw.z * qscale), static_cast<_Float16>(qraw.w * qscale)};
        if (qj >= group) h = half4{0, 0, 0, 0};
        *reinterpret_cast<half4 *>(sm_q + qj * kQStride + c4) = h;
    }
    uint2 packed{0u, 0u};
    if (fused && wave == 0) {
        if constexpr (PREP) {  // (the upper half's row is the values', which stay as they are)
            const float4 k = prep_chunk(nraw, fold.prep_k_weight != nullptr, wk, fold.prep_eps, c4, lane, prot, pinter, trig);
            if (lane < 32) nraw = k;
        }
        const uint32_t h0 = f32_to_f16_bits(nraw.x), h1 = f32_to_f16_bits(nraw.y);
        const uint32_t h2 = f32_to_f16_bits(nraw.z), h3 = f32_to_f16_bits(nraw.w);
        packed = uint2{h0 | (h1 << 16), h2 | (h3 << 16)};
        *reinterpret_cast<uint2 *>(sm_new + (lane >> 5) * kD + c4) = packed;
    }
    lds_barrier();
    half8 qb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) qb[k] = *reinterpret_cast<const half8 *>(sm_q + jl * kQStride + k * 32 + g * 8);

    const uint32_t new_kb = pos / kBlockKeys, kk = pos % kBlockKeys;
    const uint32_t lo = RING ? lowest_visible(pos, p.window, item.kv_lo) : 0;
    float sc[R][8], mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves, key_base = kb * kBlockKeys + g * 8;
        if (fused && kb == new_kb) {
            // Keys: lane (g, i) holds row i of tile t; the new key is row i_new of tile t_new.
            const uint32_t t_new = (kk >> 2) & 1, i_new = (kk >> 3) * 4 + (kk & 3);
            if (jl == i_new) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const half8 h = *reinterpret_cast<const half8 *>(sm_new + s * 32 + g * 8);
                    if (t_new == 0) bk[r][0][s] = h; else bk[r][1][s] = h;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            floatx4 s = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < 4; ++k) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(bk[r][t][k], qb[k], s, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[r][t * 4 + e] = PREP ? s[e] : s[e] * score_scale;
        }
        if (softcap > 0.0f) {
            const float inv_cap = 1.0f / softcap;
#pragma unroll
            for (int e = 0; e < 8; ++e) sc[r][e] = softcap_log2(sc[r][e], softcap, inv_cap);
        }
        // Keys the query does not see (and blocks beyond the last) weigh nothing; their values leave the product too.
        if ((kb + 1) * kBlockKeys > pos + 1 || (RING && kb * kBlockKeys < lo)) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (key_base + e > pos || (RING && key_base + e < lo)) sc[r][e] = -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sc[r][e]);
    }
    mx = column_max4(mx);
    // (Nothing finite in sight: -inf weighs zero against a reference of zero, and a NaN score, which the maximum passes
    // over as the reference's comparison does, stays NaN.)
    const float m_ref = mx == -INFINITY ? 0.0f : mx;
    float sum = 0.0f;
    floatx4 o[kT];
#pragma unroll
    for (int c = 0; c < kT; ++c) o[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves, key_base = kb * kBlockKeys + g * 8;
        if (kb >= kb_end) break;
        half8 pb;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float pe = fast_exp2(sc[r][e] - m_ref);
            sum += pe;
            pb[e] = static_cast<_Float16>(pe);
        }
        if (fused && kb == new_kb && g == (kk >> 3)) {
            // Values: lane (g, jl) holds keys g*8 .. g*8+7 of a channel; half kk % 8 is replaced through a mask.
            const u32x4 at = first_halves((kk & 7u) + 1) & ~first_halves(kk & 7u);
#pragma unroll
            for (int c = 0; c < kT; ++c) {
                const uint32_t h = reinterpret_cast<const uint16_t *>(sm_new)[kD + (part * kT + c) * 16 + jl], both = h | (h << 16);
                const u32x4 old = __builtin_bit_cast(u32x4, bv[r][c]);
                bv[r][c] = __builtin_bit_cast(half8, (old & ~at) | (u32x4{both, both, both, both} & at));
            }
        }
        if ((kb + 1) * kBlockKeys > pos + 1 || (RING && kb * kBlockKeys < lo)) {
            const uint32_t end = min(pos + 1 - min(pos + 1, key_base), 8u);  // this lane's keys [first, end) stay
            const uint32_t first = RING ? min(lo - min(lo, key_base), 8u) : 0u;
            const u32x4 keep = first_halves(end) & ~first_halves(first);
#pragma unroll
            for (int c = 0; c < kT; ++c) bv[r][c] = keep_halves(bv[r][c], keep);
        }
#pragma unroll
        for (int c = 0; c < kT; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[r][c], pb, o[c], 0, 0, 0);
    }
    const float l_wave = column_sum4(sum);
    if (g == 0) {
        sm_m[wave * 16 + jl] = mx;
        sm_l[wave * 16 + jl] = l_wave;
    }
#pragma unroll
    for (int c = 0; c < kT; ++c) *reinterpret_cast<floatx4 *>(sm_o + ((wave * kT + c) * 64 + lane) * 4) = o[c];
    lds_barrier();
    float mw[kWaves], lw[kWaves], ow[kF][kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        mw[w] = sm_m[w * 16 + fcol];
        lw[w] = sm_l[w * 16 + fcol];
#pragma unroll
        for (int u = 0; u < kF; ++u) ow[u][w] = sm_o[w * kT * 256 + u * 512 + (P == 8 ? tid & 255 : tid)];
    }
    float M = mw[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) M = fmaxf(M, mw[w]);
    float L = 0.0f, acc[kF];
#pragma unroll
    for (int u = 0; u < kF; ++u) acc[u] = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const float wgt = mw[w] == -INFINITY ? 0.0f : fast_exp2(mw[w] - M);
        L = fmaf(lw[w], wgt, L);
#pragma unroll
        for (int u = 0; u < kF; ++u) acc[u] = fmaf(ow[u][w], wgt, acc[u]);
    }
    if (fcol < group && (P != 8 || tid < 256)) {
        const float inv = __builtin_amdgcn_rcpf(L);
#pragma unroll
        for (int u = 0; u < kF; ++u) {
            float y = acc[u] * inv;
            if (PREP && fold.gate) y *= sigmoid_fast(gt[u]);
            p.out[out_at + u * 32] = y;
        }
    }
    // The new row goes to the planes as append lays it out; nothing in this launch reads it from there.
    if (fused && wave == 0 && part == 0) {
        uint32_t nsb = new_kb;
        if (RING) nsb %= ring_blocks;
        const uint64_t blk = uint64_t(nsb) * (kBlockKeys * kD);
        if (lane < 32) {
            const uint32_t kt = (kk >> 2) & 1, ki = (kk >> 3) * 4 + (kk & 3);
            *reinterpret_cast<uint2 *>(kplane + blk + ((kt * 16 + (c4 >> 3)) * 16 + ki) * 8 + (c4 & 7)) = packed;
        } else {
            uint16_t *vd = vplane + blk + c4 * kBlockKeys + kk;
            vd[0] = uint16_t(packed.x);
            vd[kBlockKeys] = uint16_t(packed.x >> 16);
            vd[2 * kBlockKeys] = uint16_t(packed.y);
            vd[3 * kBlockKeys] = uint16_t(packed.y >> 16);
        }
    }
}
template <int N, bool RING, int P, int R>
__global__ __launch_bounds__(kWaves * 64) void attn_whole_f16_kernel(AttnParams p, AttnBatchT<N> b) {
    attn_whole_f16_body<N, RING, false, P, R>(p, b, FoldedParams{});
}
template <int N, bool RING, int P, int R>
__global__ __launch_bounds__(kWaves * 64) void attn_whole_f16_prep_kernel(AttnParams p, AttnBatchT<N> b, FoldedParams f) {
    attn_whole_f16_body<N, RING, true, P, R>(p, b, f);
}

}  // namespace

hipError_t launch_attn_whole_f16(const AttnParams &p, const AttnBatch &b, hipStream_t stream, const FoldedParams *prepares) {
    if (b.total_blocks == 0) return hipSuccess;
    uint32_t most = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        const AttnItem &it = b.item[i];
        if (it.rows != 1 || it.pos0 + 1 != it.kv_len || it.splits != 1) return hipErrorInvalidValue;
        most = std::max(most, item_block_count(it));
    }
    const uint32_t rounds = (most + kWaves - 1) / kWaves;
    if (rounds > kWholeMostBlocks / kWaves || (b.parts != 2 && b.parts != 4 && b.parts != 8)) return hipErrorInvalidValue;  // (the planner asks for no more)
#define ITAK_WHOLE(P, R)                                                                                             \
    do {                                                                                                             \
        if (prepares && p.ring_blocks)                                                                               \
            launch_kernel(attn_whole_f16_prep_kernel<N, true, P, R>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<N>(b), *prepares); \
        else if (prepares)                                                                                           \
            launch_kernel(attn_whole_f16_prep_kernel<N, false, P, R>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<N>(b), *prepares); \
        else if (p.ring_blocks)                                                                                      \
            launch_kernel(attn_whole_f16_kernel<N, true, P, R>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<N>(b)); \
        else                                                                                                         \
            launch_kernel(attn_whole_f16_kernel<N, false, P, R>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<N>(b)); \
    } while (0)
#define ITAK_WHOLE_R(P)                                                  \
    do {                                                                 \
        if (rounds <= 1) ITAK_DISPATCH_BATCH(b.n, ITAK_WHOLE(P, 1));     \
        else if (rounds == 2) ITAK_DISPATCH_BATCH(b.n, ITAK_WHOLE(P, 2)); \
        else ITAK_DISPATCH_BATCH(b.n, ITAK_WHOLE(P, 3));                 \
    } while (0)
    if (b.parts == 8) ITAK_WHOLE_R(8);
    else if (b.parts == 4) ITAK_WHOLE_R(4);
    else ITAK_WHOLE_R(2);
#undef ITAK_WHOLE_R
#undef ITAK_WHOLE
    return hipGetLastError();
}

}  // namespace itak
