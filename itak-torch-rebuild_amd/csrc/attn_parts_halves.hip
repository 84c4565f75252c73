// GQA flash-decode for gfx950 on f16 pools at the head dims attn_splitk_halves_kernel serves (blocked planes, head_dim a
// multiple of 16): one row per sequence, while the work is at most one workgroup per compute unit.
//
// The work is cut as in attn_whole_f16.hip: each workgroup of a (slot, KV head) works out all scores and the output of KT of
// its channel tiles, eight wavefronts of up to four blocks each, every load asked for before anything is waited for.
// Contexts beyond are cut into runs of eight blocks, one a wavefront, and merged by a second launch. The
// arithmetic is attn_splitk_halves_kernel's (attn_splitk_any.hip): queries and weights as three halves each, a
// wavefront whose sums come out not finite walks its keys again on the f32 pipe. What cost that kernel's steps
// most, beside the merge launch, was done once per wavefront there and is done once per workgroup here: the queries' split
// into halves (64 channels a lane at head_dim 256; 4 or 8 here, shared through LDS), and the new row, which was stored,
// waited for and read back and is patched into the operands now.
// 32 Q / 4 KV heads, us a layer, attn_splitk_halves_kernel whole or split -> this. Whole, one slot at 60 / 200 / 400 / 700
// positions, head_dim 64 4.9 / 5.6 / 6.6 / 7.0 -> 4.2 / 4.4 / 5.2 / 6.0, head_dim 80 5.2 / 6.4 / 7.7 / 7.5 -> 4.4 / 4.6 / 5.5 / 6.5,
// head_dim 112 5.8 / 7.4 / 8.9 / 8.2 -> 4.6 / 4.8 / 6.0 / 7.3; at 60 / 200 / 400 head_dim 192 8.0 / 9.4 / 10.4 ->
// 5.3 / 5.5 / 7.5, head_dim 256 9.6 / 11.5 / 12.0 -> 5.7 / 5.9 / 8.6; 8 slots at 200 / 700, head_dim 80 6.9 / 9.5 -> 5.0 / 7.2.
// Split, one slot at 1,500 / 3,000, head_dim 64 7.0 / 7.5 -> 6.5 / 7.0, head_dim 80 8.1 / 8.5 -> 7.2 / 7.6, head_dim 112 8.9 / 9.1 ->
// 7.7 / 7.9, head_dim 256 12.5 / 12.8 -> 8.6 / 9.1; 4 slots at 1,500 head_dim 80 9.2 -> 8.1, head_dim 192 12.9 -> 11.3; 8 slots
// at 1,500 head_dim 96 11.1 -> 9.7.
// What bounds it now: launch and first trips to memory, 2.5 us, the products of eight wavefronts on one compute unit's
// matrix pipes (0.3 us a round at head_dim 80, three for one with f32's precision), the keys each part reads, and the merge.
//
// Semantics: gqa_attention in crates/attention/src/attention.rs:104-215, softcap as
// crates/torch-math/src/logits.rs:26-37. Partials are in the log2 domain.
#include "attn_splitk_rows_kernel.h"

#include <math.h>

#include <algorithm>

namespace itak {

namespace {

constexpr int kWaves = 8;

// The largest over the 32 lanes that share a query vector.
__device__ __forceinline__ float row_max32(float v) {
    v = fmaxf(v, dpp_lane<0xB1>(v));   // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_lane<0x4E>(v));   // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_lane<0x141>(v));  // row_half_mirror
    v = fmaxf(v, dpp_lane<0x140>(v));  // row_mirror
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// DP: head_dim rounded up to a multiple of 32; KT: channel tiles of a workgroup; R: blocks of a wavefront; SPLIT: contexts may be
// cut (without it the whole forms were 2 % slower).
template <int DP, int KT, int R, bool SPLIT, int N>
__global__ __launch_bounds__(kWaves * 64) void attn_parts_halves_kernel(AttnParams p, AttnBatchT<N> b,
                                                                        uint32_t total_partials) {
    constexpr int kS = DP / 32;       // steps of a key row
    constexpr int kStride = DP + 8;   // LDS row stride of the staged queries (halves)
    constexpr int kQ = DP > 128 ? 2 : 1;  // pieces of four channels of a query a thread stages
    __shared__ __attribute__((aligned(16))) _Float16 sm_q[3][16 * kStride];
    __shared__ __attribute__((aligned(16))) _Float16 sm_new[2 * DP];  // the new K row, then the new V row
    __shared__ float sm_scale[16], sm_m[kWaves * 16], sm_l[kWaves * 16];
    __shared__ __attribute__((aligned(16))) float sm_o[kWaves * KT * 256];  // [wave][tile][lane][row of the lane]

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t g = lane >> 4, jl = lane & 15;
    const uint32_t D = p.g.head_dim, chunks = D / 8, quads = D / 4;

    const AttnItem item = b.of_block(blockIdx.x);
    const uint32_t local = blockIdx.x - item.block0, heads = p.g.kv_heads, group = p.group;
    // Part after part, and within one split after split, so that with a multiple of eight (KV head, split) pairs the parts of one
    // run on one compute die.
    const uint32_t pairs = SPLIT ? heads * item.splits : heads, part = pairs > 1 ? __umulhi(local, item.splits_magic) : local;
    uint32_t kv_head = local - part * pairs, split = 0;
    if (SPLIT && item.splits > 1) {  // (a thousand pairs at most: a float holds the quotient)
        split = __builtin_amdgcn_readfirstlane(int((float(kv_head) + 0.5f) * __builtin_amdgcn_rcpf(float(heads))));
        kv_head -= split * heads;
    }

    uint16_t *kplane = static_cast<uint16_t *>(const_cast<void *>(p.layer_base)) + item.slot * p.g.slot_stride +
                       kv_head * p.g.head_stride;
    uint16_t *vplane = kplane + p.g.side_stride;
    const uint32_t ring_blocks = p.ring_blocks;
    const uint32_t pos = min(item.pos0, item.kv_len - 1);  // the newest position the query sees, and the oldest
    const uint32_t lo = lowest_visible(item.pos0, p.window, item.kv_lo);
    const uint32_t run = SPLIT ? item.keys_per_split / kBlockKeys : 0, kb_begin = lo / kBlockKeys + split * run;
    const uint32_t kb_end = SPLIT ? min(pos / kBlockKeys + 1, kb_begin + run) : pos / kBlockKeys + 1;
    auto block_at = [&](uint32_t kb) { return uint64_t(ring_blocks ? kb % ring_blocks : kb) * (kVBlock * D); };

    // ---- every load: the new row (its keys' pieces, then its values'), the queries (32 threads a vector; vectors beyond
    // the group re-read the last), the wavefront's blocks wave, wave + 8, .. from the first. In place of one beyond the last
    // every lane loads the same 16 bytes, one line a load.
    const bool fused = p.k_new != nullptr;
    const uint32_t np = min(tid, 2 * quads - 1), nside = np >= quads ? 1u : 0u, nc4 = (np - nside * quads) * 4;
    const float *nsrc = (nside ? p.v_new : p.k_new) + (uint64_t(item.q_row0) * heads + kv_head) * D + nc4;
    const floatx4 nraw = *reinterpret_cast<const floatx4 *>(fused ? nsrc : p.q);
    const uint32_t qj = tid >> 5, qc = tid & 31;
    const float *qrow = p.q + (uint64_t(item.q_row0) * p.q_heads + kv_head * group) * D;
    floatx4 x[kQ];
#pragma unroll
    for (int u = 0; u < kQ; ++u)
        x[u] = *reinterpret_cast<const floatx4 *>(qrow + min(qj, group - 1) * D + 4 * min(qc + 32u * u, quads - 1));
    half8 k[R][2][kS], v[R][KT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves;
        const bool has = kb < kb_end;
        const uint16_t *kblk = kplane + block_at(has ? kb : kb_begin);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < kS; ++s)
                k[r][t][s] = *reinterpret_cast<const half8 *>(
                    kblk + (has ? ((t * chunks + min(4u * s + g, chunks - 1)) * 16 + jl) * 8 : 0));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves;
        const bool has = kb < kb_end;
        const uint16_t *vblk = vplane + block_at(has ? kb : kb_begin);
#pragma unroll
        for (int c = 0; c < KT; ++c)
            v[r][c] = *reinterpret_cast<const half8 *>(
                vblk + (has ? min((part * KT + c) * 16 + jl, D - 1) * kVBlock + 8 * g : 0));
    }
    __builtin_amdgcn_sched_barrier(0);

    const float softcap = p.softcap;
    const float inv_cap = softcap > 0.0f ? 1.0f / softcap : 0.0f;
    const float qscale = softcap > 0.0f ? p.scale : p.scale * kLog2e;
    {
        // A vector as three halves, times the power of two that brings its largest below 2^15.
        float most = 0.0f;
#pragma unroll
        for (int u = 0; u < kQ; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (qc + 32u * u >= quads || qj >= group) x[u][e] = 0.0f;
                most = fmaxf(most, fabsf(x[u][e]));
            }
        most = row_max32(most);
        const int up = 15 - __builtin_amdgcn_frexp_expf(most);  // (0 for zero and for what is not finite: 2^15)
#pragma unroll
        for (int u = 0; u < kQ; ++u) {
            half4 h0, h1, h2;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                _Float16 a, c, d;
                split3(ldexpf(x[u][e], up), a, c, d);
                h0[e] = a, h1[e] = c, h2[e] = d;
            }
            const uint32_t at = qj * kStride + 4 * (qc + 32u * u);
            if (4 * (qc + 32u * u) < DP) {
                *reinterpret_cast<half4 *>(&sm_q[0][at]) = h0;
                *reinterpret_cast<half4 *>(&sm_q[1][at]) = h1;
                *reinterpret_cast<half4 *>(&sm_q[2][at]) = h2;
            }
        }
        if (qc == 0) sm_scale[qj] = ldexpf(qscale, -up);
    }
    uint2 packed{0u, 0u};
    if (fused && tid < 2 * quads) {
        packed = uint2{f32_to_f16_bits(nraw[0]) | uint32_t(f32_to_f16_bits(nraw[1])) << 16,
                       f32_to_f16_bits(nraw[2]) | uint32_t(f32_to_f16_bits(nraw[3])) << 16};
        *reinterpret_cast<uint2 *>(sm_new + nside * DP + nc4) = packed;
    }
    lds_barrier();
    const float colscale = sm_scale[jl];
    auto query = [&](int h, int s) { return *reinterpret_cast<const half8 *>(&sm_q[h][jl * kStride + 32 * s + 8 * g]); };
    half8 q[DP <= 128 ? kS : 1][3];
    if constexpr (DP <= 128) {
#pragma unroll
        for (int s = 0; s < kS; ++s)
#pragma unroll
            for (int h = 0; h < 3; ++h) q[s][h] = query(h, s);
    }

    const uint32_t new_kb = fused ? item.pos0 / kBlockKeys : 0xffffffffu, kk = item.pos0 % kBlockKeys;
    const uint32_t t_new = (kk >> 2) & 1, i_new = (kk >> 3) * 4 + (kk & 3);  // the new key's tile and row
    float sc[R][8], mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves, key0 = kb * kBlockKeys + 8 * g;
        if (kb == new_kb && jl == i_new) {
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                const half8 h = *reinterpret_cast<const half8 *>(sm_new + min(4u * s + g, chunks - 1) * 8);
                if (t_new == 0) k[r][0][s] = h; else k[r][1][s] = h;
            }
        }
        floatx4 acc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < kS; ++s) {
            half8 qs[3];
#pragma unroll
            for (int h = 0; h < 3; ++h) {
                if constexpr (DP <= 128) qs[h] = q[s][h]; else qs[h] = query(h, s);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                // (Only the last step can lie beyond head_dim, and then in half of the lanes.)
                if (s == kS - 1 && 4u * s + g >= chunks) k[r][t][s] = half8{};
#pragma unroll
                for (int h = 2; h >= 0; --h) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k[r][t][s], qs[h], acc[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sc[r][e] = acc[e / 4][e % 4] * colscale;
            if (softcap > 0.0f) sc[r][e] = softcap_log2(sc[r][e], softcap, inv_cap);
        }
        // Keys the query does not see score nothing, and neither does what a wavefront loaded in place of a block beyond its
        // run: whole contexts' and the last run's end at `pos`, the others' before it. (As the end that keys are compared with it
        // costs nothing, one slot at 1,500, head_dim 64 / 80 / 256, 6.9 / 7.4 / 8.6 us a layer; as a condition beside them 0.2 us.)
        const uint32_t end = SPLIT && kb >= kb_end ? 0 : pos + 1;
        if ((kb + 1) * kBlockKeys > end || kb * kBlockKeys < lo) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (key0 + e >= end || key0 + e < lo) sc[r][e] = -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sc[r][e]);
    }
    float m_run = lanes4_max(mx), l_run = 0.0f;
    floatx4 o[KT];
#pragma unroll
    for (int c = 0; c < KT; ++c) o[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t kb = kb_begin + wave + r * kWaves, key0 = kb * kBlockKeys + 8 * g;
        if (kb >= kb_end) break;
        half8 w[3];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            // (Nothing finite in sight: -inf weighs zero against a reference of zero, and a NaN score stays NaN.)
            const float pe = fast_exp2(sc[r][e] - (m_run == -INFINITY ? 0.0f : m_run) + kWeightShift);
            l_run += pe;
            _Float16 h0, h1, h2;
            split3(pe, h0, h1, h2);
            w[0][e] = h0, w[1][e] = h1, w[2][e] = h2;
        }
        if (kb == new_kb && g == (kk >> 3)) {
            const u32x4 at = first_halves((kk & 7u) + 1) & ~first_halves(kk & 7u);
#pragma unroll
            for (int c = 0; c < KT; ++c) {
                const uint32_t h = reinterpret_cast<const uint16_t *>(sm_new)[DP + min((part * KT + c) * 16 + jl, D - 1)];
                const uint32_t both = h | (h << 16);
                const u32x4 old = __builtin_bit_cast(u32x4, v[r][c]);
                v[r][c] = __builtin_bit_cast(half8, (old & ~at) | (u32x4{both, both, both, both} & at));
            }
        }
        // A row the query does not see may hold anything: kept out of P.V even as 0 * x.
        if ((kb + 1) * kBlockKeys > pos + 1 || kb * kBlockKeys < lo) {
            const u32x4 keep = first_halves(min(pos + 1 - min(pos + 1, key0), 8u)) & ~first_halves(min(lo - min(lo, key0), 8u));
#pragma unroll
            for (int c = 0; c < KT; ++c) v[r][c] = keep_halves(v[r][c], keep);
        }
#pragma unroll
        for (int c = 0; c < KT; ++c)
#pragma unroll
            for (int h = 2; h >= 0; --h) o[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v[r][c], w[h], o[c], 0, 0, 0);
    }

    float all = l_run;
#pragma unroll
    for (int c = 0; c < KT; ++c) {
        all += (o[c][0] + o[c][1]) + (o[c][2] + o[c][3]);
        *reinterpret_cast<floatx4 *>(sm_o + ((wave * KT + c) * 64 + lane) * 4) = o[c];
    }
    // Sums that are not finite: again on the f32 pipe (an infinite row times halves of which one is zero or of the other sign
    // is NaN where the product is not), an output tile at a time. Cold and small rather than fast.
    if (__builtin_amdgcn_ballot_w64(!(fabsf(all) < INFINITY)) != 0) {
        const float *qp = qrow + min(jl, group - 1) * D;
#pragma unroll 1
        for (int c = 0; c < KT; ++c) {
            const uint32_t ch_out = min((part * KT + c) * 16 + jl, D - 1);
            floatx4 out = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            m_run = -INFINITY;
            l_run = 0.0f;
#pragma unroll 1
            for (uint32_t kb = kb_begin + wave; kb < kb_end; kb += kWaves) {
                const uint32_t key0 = kb * kBlockKeys;
                const uint64_t at = block_at(kb);
                floatx4 acc[2] = {};
#pragma unroll 1
                for (uint32_t ch = g; ch < D; ch += 4) {
                    const float qv = jl < group ? qp[ch] * qscale : 0.0f;
#pragma unroll
                    for (uint32_t t = 0; t < 2; ++t) {
                        const bool is_new = kb == new_kb && t == t_new && jl == i_new;
                        const uint16_t bits = is_new ? reinterpret_cast<const uint16_t *>(sm_new)[ch]
                                                     : kplane[at + ((t * chunks + ch / 8) * 16 + jl) * 8 + ch % 8];
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(float(__builtin_bit_cast(_Float16, bits)), qv, acc[t], 0, 0, 0);
                    }
                }
                float s8[8], top = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float s = acc[e / 4][e % 4];
                    if (softcap > 0.0f) s = softcap_log2(s, softcap, inv_cap);
                    const uint32_t kp = key0 + 8 * g + e;
                    s8[e] = kp > pos || kp < lo ? -INFINITY : s;
                    top = fmaxf(top, s8[e]);
                }
                const float m_new = fmaxf(m_run, lanes4_max(top)), ref = m_new == -INFINITY ? 0.0f : m_new;
                const float alpha = m_run == -INFINITY ? (m_new == -INFINITY ? 1.0f : 0.0f) : fast_exp2(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
                out *= alpha;
                const uint16_t *vv = vplane + at + ch_out * kVBlock + 8 * g;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float pe = fast_exp2(s8[e] - ref + kWeightShift);
                    l_run += pe;
                    const uint32_t kp = key0 + 8 * g + e;
                    const uint16_t bits = fused && kp == item.pos0 ? reinterpret_cast<const uint16_t *>(sm_new)[DP + ch_out] : vv[e];
                    const float val = kp <= pos && kp >= lo ? float(__builtin_bit_cast(_Float16, bits)) : 0.0f;
                    out = __builtin_amdgcn_mfma_f32_16x16x4f32(val, pe, out, 0, 0, 0);
                }
            }
            *reinterpret_cast<floatx4 *>(sm_o + ((wave * KT + c) * 64 + lane) * 4) = out;
        }
    }

    const float l_col = lanes4_sum(l_run);
    if (g == 0) {
        sm_m[wave * 16 + jl] = m_run;
        sm_l[wave * 16 + jl] = l_col;
    }
    lds_barrier();
    // Value tid + 64 kWaves u of the part's outputs, [tile][lane][row of the lane].
    static_assert(KT == 1 || KT % 2 == 0, "every thread has as many values");
    constexpr int kValues = KT * 256, kF = (KT + 1) / 2;
    const bool final_out = !SPLIT || item.splits == 1;
    if (wave * 64 >= kValues) return;
    const uint32_t fcol = (tid >> 2) & 15, fch = part * KT * 16 + (tid >> 8) * 16 + ((tid >> 6) & 3) * 4 + (tid & 3);
    float mw[kWaves], lw[kWaves], ow[kF][kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        mw[w] = sm_m[w * 16 + fcol];
        lw[w] = sm_l[w * 16 + fcol];
#pragma unroll
        for (int u = 0; u < kF; ++u) ow[u][w] = sm_o[w * kValues + u * kWaves * 64 + tid];
    }
    float M = mw[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) M = fmaxf(M, mw[w]);
    float L = 0.0f, fin[kF];
#pragma unroll
    for (int u = 0; u < kF; ++u) fin[u] = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const float wgt = mw[w] == -INFINITY ? 0.0f : fast_exp2(mw[w] - M);
        L = fmaf(lw[w], wgt, L);
#pragma unroll
        for (int u = 0; u < kF; ++u) fin[u] = fmaf(ow[u][w], wgt, fin[u]);
    }
    if (fcol < group) {
        const uint32_t head = kv_head * group + fcol;
        const uint64_t ps = item.ws0 + uint64_t(head) * item.splits + split;
        const float post = final_out ? 1.0f / L : 1.0f;
        float *dst = final_out ? p.out + (uint64_t(item.q_row0) * p.q_heads + head) * D : p.ws + ps * D;
#pragma unroll
        for (int u = 0; u < kF; ++u)
            if (fch + 4 * kWaves * u < D) dst[fch + 4 * kWaves * u] = fin[u] * post;
        if (!final_out && part == 0 && tid < 64 && (tid & 3) == 0)
            *reinterpret_cast<float2 *>(p.ws + uint64_t(total_partials) * D + ps * 2) = make_float2(M, L);
    }
    // The new row goes to the planes as append lays it out; nothing in this launch reads it from there.
    if (fused && part == 0 && (!SPLIT || new_kb - kb_begin < kb_end - kb_begin) && tid < 2 * quads) {
        const uint64_t blk = block_at(new_kb);
        if (nside == 0) {
            *reinterpret_cast<uint2 *>(kplane + blk + ((t_new * chunks + nc4 / 8) * 16 + i_new) * 8 + nc4 % 8) = packed;
        } else {
            uint16_t *vd = vplane + blk + nc4 * kVBlock + kk;
            vd[0] = uint16_t(packed.x);
            vd[kVBlock] = uint16_t(packed.x >> 16);
            vd[2 * kVBlock] = uint16_t(packed.y);
            vd[3 * kVBlock] = uint16_t(packed.y >> 16);
        }
    }
}

// Channel tiles a workgroup may have: one, two, four or all up to head_dim 128; two, four or eight beyond, where the keys
// are the larger part of what a workgroup reads.
uint32_t next_tiles(uint32_t d, uint32_t kt) {
    if (kt == 0) return d <= 128 ? 1 : 2;
    if (kt < (d <= 128 ? 4u : 8u)) return 2 * kt;
    const uint32_t all = (d + 31) / 32 * 2;
    return d <= 128 && kt < all ? all : 0;
}

}  // namespace

// Takes a batch of one-row steps when every workgroup has a compute unit to itself: whole contexts, or runs of eight blocks, one
// for each wavefront, with as few channel tiles a workgroup as that allows. (More workgroups than compute units lose to
// attn_splitk_halves_kernel: 8 slots at 3,000, head_dim 80, 384 workgroups of all tiles 13.1 against 12.6; runs of 10 or 12 blocks on
// as many wavefronts are no faster than that kernel either, 10.2 against 10.3 where runs of eight take 9.1.)
bool attn_parts_halves_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, uint32_t *partials) {
    const uint32_t d = g.head_dim, tiles = d / 16;
    if (!g.v_block || d % 16 != 0 || d > 256 || q_heads / g.kv_heads > 16) return false;
    uint32_t most = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        if (b.item[i].rows != 1) return false;
        most = std::max(most, item_block_count(b.item[i]));
    }
    const uint64_t units = uint64_t(g.kv_heads) * b.n, cus = compute_units();
    auto groups_at = [&](uint32_t run, uint32_t kt) {
        uint64_t pairs = 0;
        for (uint32_t i = 0; i < b.n; ++i)
            pairs += uint64_t(g.kv_heads) * std::max((item_block_count(b.item[i]) + run - 1) / run, 1u);
        return pairs * ((tiles + kt - 1) / kt);
    };
    uint32_t T = 0;
    auto fits = [&](uint32_t run, uint32_t most_kt) {
        for (uint32_t kt = next_tiles(d, 0); kt && kt <= most_kt; kt = next_tiles(d, kt))
            if (groups_at(run, kt) <= cus) {
                b.parts = kt;
                T = run;
                return true;
            }
        return false;
    };
    // Whole first: two rounds above head_dim 128 (a third spills), three below; a fourth where a merge has many outputs, from 16 units on, at
    // head_dim 64 before and at others after the cut. Below 16 units the cut wins from the fourth on: one slot at 800,
    // head_dim 64 / 112, split 6.6 / 7.2, whole 6.6 / 8.3. Cut second, where a context has a fourth round: the general forms leave up
    // to 24 blocks whole from 16 units on, and better so (24 slots at 400, head_dim 80, 8.4 whole, 9.4 split).
    const uint32_t whole_kt = d <= 128 ? 2 : 4, rounds = (most + kWaves - 1) / kWaves;
    const bool many = d <= 128 && units >= 16;
    const uint32_t whole_rounds = d > 128 ? 2 : many && d <= 64 ? 4 : 3;
    if (!(rounds <= whole_rounds && fits(most, whole_kt)) && !(rounds > (many ? 3u : 1u) && fits(kWaves, 16)) &&
        !(many && rounds <= 4 && fits(most, whole_kt)))
        return false;
    uint32_t block0 = 0, ws0 = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        AttnItem &it = b.item[i];
        const uint32_t nblocks = std::max(item_block_count(it), 1u);
        it.splits = (nblocks + T - 1) / T;
        const uint32_t run = (nblocks + it.splits - 1) / it.splits;
        it.splits = (nblocks + run - 1) / run;
        it.keys_per_split = run * kBlockKeys;
        const uint64_t pairs = uint64_t(g.kv_heads) * it.splits;
        it.splits_magic = pairs > 1 ? uint32_t(((uint64_t(1) << 32) + pairs - 1) / pairs) : 0;
        it.block0 = block0;
        it.ws0 = ws0;
        block0 += g.kv_heads * ((tiles + b.parts - 1) / b.parts) * it.splits;
        if (it.splits > 1) ws0 += q_heads * it.splits;
    }
    b.total_blocks = block0;
    b.rows_per_block = 0;
    *partials = ws0;
    return true;
}

hipError_t launch_attn_parts_halves(const AttnParams &p, const AttnBatch &b, uint32_t total_partials, hipStream_t stream) {
    uint32_t most = 1;
    bool split = false;
    for (uint32_t i = 0; i < b.n; ++i) {
        most = std::max(most, b.item[i].keys_per_split / kBlockKeys);
        split = split || b.item[i].splits > 1;
    }
    const uint32_t rounds = (most + kWaves - 1) / kWaves, d = p.g.head_dim;
#define ITAK_PARTS(DP, KT, R, SPLIT)                                                                                   \
    do {                                                                                                               \
        if (b.n <= 8)                                                                                                  \
            launch_kernel(attn_parts_halves_kernel<DP, KT, R, SPLIT, 8>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<8>(b), total_partials); \
        else                                                                                                           \
            launch_kernel(attn_parts_halves_kernel<DP, KT, R, SPLIT, 64>, b.total_blocks, kWaves * 64, 0, stream, p, AttnBatchT<64>(b), total_partials); \
        return hipGetLastError();                                                                                      \
    } while (0)
// (Split runs are one round; WHOLE = the rounds of whole contexts, of which the forms of most tiles have none.)
#define ITAK_PARTS_R(DP, KT, WHOLE)                                              \
    if (b.parts == KT) {                                                         \
        if (split && rounds == 1) ITAK_PARTS(DP, KT, 1, true);                   \
        if constexpr (WHOLE >= 2) {                                              \
            if (!split && rounds == 1) ITAK_PARTS(DP, KT, 1, false);             \
            if (!split && rounds == 2) ITAK_PARTS(DP, KT, 2, false);             \
        }                                                                        \
        if constexpr (WHOLE >= 4) {                                              \
            if (!split && rounds == 3) ITAK_PARTS(DP, KT, 3, false);             \
            if (!split && rounds == 4) ITAK_PARTS(DP, KT, 4, false);             \
        }                                                                        \
    }
#define ITAK_PARTS_T(DP)                                                 \
    do {                                                                 \
        if constexpr (DP <= 128) {                                       \
            ITAK_PARTS_R(DP, 1, 4)                                       \
            ITAK_PARTS_R(DP, 2, 4)                                       \
            ITAK_PARTS_R(DP, 4, 0)                                       \
            if constexpr (DP > 64) ITAK_PARTS_R(DP, (DP / 16), 0)        \
        } else {                                                         \
            ITAK_PARTS_R(DP, 2, 2)                                       \
            ITAK_PARTS_R(DP, 4, 2)                                       \
            ITAK_PARTS_R(DP, 8, 0)                                       \
        }                                                                \
    } while (0)
    switch ((d + 31) / 32) {
        case 1: ITAK_PARTS_T(32); break;
        case 2: ITAK_PARTS_T(64); break;
        case 3: ITAK_PARTS_T(96); break;
        case 4: ITAK_PARTS_T(128); break;
        case 5: ITAK_PARTS_T(160); break;
        case 6: ITAK_PARTS_T(192); break;
        case 7: ITAK_PARTS_T(224); break;
        default: ITAK_PARTS_T(256); break;
    }
#undef ITAK_PARTS_T
#undef ITAK_PARTS_R
#undef ITAK_PARTS
    return hipErrorInvalidValue;  // (the planner asks for no others)
}

}  // namespace itak
