// GQA attention for gfx950 at the head dims the other matrix kernels are not written for: f16 pools
// at any head_dim that is a multiple of four (and any GQA group), f32 pools at head dims other than
// 64 and 128. Decode steps, blocks and chunks, split over the context. Queries and softmax weights
// keep f32's precision, so that an f16 pool gives here what f32 arithmetic over its rows gives. A
// short step's new rows are appended by the same launch.
//
// The shape of the work is attn_splitk_rows_kernel's (a workgroup of four or eight wavefronts = item, KV
// head, tile of 16 query vectors, run of 32-key blocks; a private online softmax per wavefront,
// one merge through LDS) and its launches are planned by the same rule. What differs is the
// operands. Which channel and which key an MFMA's k index stands for is free, and is chosen so that
// every load is one contiguous piece per lane in the layout at hand (lane = i + 16 g):
//
//   blocked f16 planes (head_dim a multiple of 16): attn_splitk_halves_kernel
//     Rows that are halves already need no f32 pipe: a float is the sum of three halves (33 bits,
//     once a power of two has brought the largest of the row to 2^14), a product of halves is exact
//     in f32, and v_mfma_f32_16x16x32_f16 does in 16 cycles what eight f32 products do in 256. So
//     Q and the softmax weights enter as three halves each, three products where one would round,
//     and every sum is f32 as before.
//     S^T tile t   lane (i, g) reads the 16-byte piece of 8 channels at chunk 4s + g of the tile's
//                  row i: the operand as it lies. Lane (j, g) receives the scores of keys 8g + 4t + r.
//     O^T tile c   lane (i, g) reads the 8 keys 8g .. 8g + 7 of channel 16c + i: the same eight
//                  keys whose weights the lane (j, g) holds. Rows of the tile are channels.
//     An infinite row times three halves of different signs, or of which one is zero, is NaN where
//     the product is not: a wavefront whose sums come out not finite walks its keys again on the
//     f32 pipe, query row by query row.
//   row-major planes (f32; f16 at other multiples of 4): attn_splitk_rows_kernel.h
//
// DP is head_dim rounded up to a multiple of 32 (blocked) or 64 (row-major); pieces beyond head_dim
// are read from the row's last valid piece and taken as zero.
//
// Bound: launch and memory latency on decode steps; on blocks the L2 that feeds a workgroup per 16
// vectors (row-major: the f32 matrix pipe, 157 TFLOP/s).
// The general VALU kernel, which these shapes took before, moves K and V through LDS as f32 and pays
// an LDS read for every multiply-add. 32 Q / 8 KV heads, f16, us a layer, append and merge included:
// head_dim 80, 8 slots of up to 1,500 rows 133 -> 13.4 (10.6 of it this kernel; 25.6 with its products
// on the f32 pipe), 2 slots of 40 rows at 2,000 27.6, a 512-row chunk over 2,000 rows 76 (247 on the f32
// pipe).
//
// Semantics: gqa_attention in crates/attention/src/attention.rs:104-215, softcap as
// crates/torch-math/src/logits.rs:26-37. Partials are in the log2 domain.
#include "attn_splitk_rows_kernel.h"

#include <math.h>

#include <algorithm>

namespace itak {

namespace {

template <int DP, int W, int N>
__global__ __launch_bounds__(W * 64, DP <= 128 ? 8 / W : 1) void attn_splitk_halves_kernel(AttnParams p, AttnBatchT<N> b,
                                                                                          uint32_t total_partials) {
    constexpr int kTiles = DP / 16;  // output tiles
    constexpr int kS = DP / 32;      // steps of a key row
    __shared__ float sm_m[W][16], sm_l[W][16];
    __shared__ float sm_o[W][kTiles][64][4];  // [wave][tile][lane][row of the lane]

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = tid >> 6, lane = tid & 63;
    const uint32_t g = lane >> 4, jl = lane & 15;
    const uint32_t D = p.g.head_dim, chunks = D / 8;

    const AttnItem item = b.of_block(blockIdx.x);
    const uint32_t local = blockIdx.x - item.block0;
    const uint32_t unit = local / item.splits, split = local % item.splits;
    const uint32_t group = p.group, nvec = item.rows * group;
    const uint32_t vtiles = (nvec + 15) / 16;
    const uint32_t kv_head = unit % p.g.kv_heads, vtile = vtiles - 1 - unit / p.g.kv_heads;
    const uint32_t row_first = (vtile * 16) / group;
    const uint32_t row_last = min(item.rows - 1, (vtile * 16 + 15) / group);

    uint16_t *kplane = static_cast<uint16_t *>(const_cast<void *>(p.layer_base)) + item.slot * p.g.slot_stride +
                       kv_head * p.g.head_stride;
    uint16_t *vplane = kplane + p.g.side_stride;

    const uint32_t ring_blocks = p.ring_blocks, window = p.window, kv_lo = item.kv_lo;
    const uint32_t nblocks = (min(item.pos0 + row_last + 1, item.kv_len) + kBlockKeys - 1) / kBlockKeys;
    const uint32_t blocks_per_split = item.keys_per_split / kBlockKeys;
    const uint32_t kb_begin = lowest_visible(item.pos0 + row_first, window, kv_lo) / kBlockKeys + split * blocks_per_split;
    const uint32_t kb_end = min(nblocks, kb_begin + blocks_per_split);

    // This lane's query vector (column jl of the tile) and what its mask and its output need.
    const uint32_t jv = vtile * 16 + jl;
    const uint32_t j = min(jv, nvec - 1);
    const uint32_t row = j / group, head = kv_head * group + j % group;
    const uint32_t colpos = min(item.pos0 + row, item.kv_len - 1);
    const uint32_t collo = lowest_visible(item.pos0 + row, window, kv_lo);
    const uint32_t tile_lo = lowest_visible(item.pos0 + row_first, window, kv_lo);
    const uint32_t tile_hi = min(item.pos0 + row_last + 1, item.kv_len);
    const float softcap = p.softcap;
    const float inv_cap = softcap > 0.0f ? 1.0f / softcap : 0.0f;
    const float qscale = softcap > 0.0f ? p.scale : p.scale * kLog2e;
    const float *qp = p.q + (uint64_t(item.q_row0 + row) * p.q_heads + head) * D;

    // Everything the first block needs is asked for before anything is waited for: the raw queries,
    // then its keys and values; later blocks' keys are asked for when the scores have used up the
    // operands of the block before, their values when its products have.
    floatx4 x[kS][2];
#pragma unroll
    for (int s = 0; s < kS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            x[s][h] = *reinterpret_cast<const floatx4 *>(qp + 8 * min(4u * s + g, chunks - 1) + 4 * h);

    half8 k[2][kS], v[kTiles];
    auto block_at = [&](uint32_t kb) { return uint64_t(ring_blocks ? kb % ring_blocks : kb) * (kVBlock * D); };
    // Fused append (p.k_new set): the wavefront that owns a block stores the new rows in it and waits
    // for the stores before it reads the block; nobody else reads these positions.
    auto append_rows = [&](uint32_t kb) {
        const uint32_t key0 = kb * kBlockKeys;
        if (p.k_new == nullptr || key0 + kBlockKeys <= item.pos0 || key0 >= item.pos0 + item.rows) return;
        uint16_t *kblk = kplane + block_at(kb), *vblk = vplane + block_at(kb);
        const uint32_t from = key0 > item.pos0 ? key0 - item.pos0 : 0;
        const uint32_t to = min(item.rows, key0 + kBlockKeys - item.pos0), quads = D / 4;
        const uint32_t pieces = (to - from) * 2 * quads;
        auto fetch = [&](uint32_t f, uint32_t &side, uint32_t &kk, uint32_t &c4) {
            const uint32_t r = from + f / (2 * quads), rest = f % (2 * quads);
            side = rest >= quads ? 1 : 0;
            c4 = (rest - side * quads) * 4;
            kk = (item.pos0 + r) % kBlockKeys;
            return *reinterpret_cast<const floatx4 *>(
                (side ? p.v_new : p.k_new) + (uint64_t(item.q_row0 + r) * p.g.kv_heads + kv_head) * D + c4);
        };
        auto place = [&](const floatx4 &y, uint32_t side, uint32_t kk, uint32_t c4) {
            uint16_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = f32_to_f16_bits(y[e]);
            if (side) {
#pragma unroll
                for (int e = 0; e < 4; ++e) vblk[(c4 + e) * kVBlock + kk] = h[e];
            } else {
                const uint32_t t = (kk >> 2) & 1, i = (kk >> 3) * 4 + (kk & 3);
                __builtin_memcpy(__builtin_assume_aligned(kblk + ((t * chunks + c4 / 8) * 16 + i) * 8 + c4 % 8, 8), h, 8);
            }
        };
        uint32_t f0 = 0;
        for (; f0 + 256 <= pieces; f0 += 256) {  // several rows: four pieces a lane under way at a time
            floatx4 y[4];
            uint32_t side[4], kk[4], c4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) y[u] = fetch(f0 + 64 * u + lane, side[u], kk[u], c4[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) place(y[u], side[u], kk[u], c4[u]);
        }
        for (uint32_t f = f0 + lane; f < pieces; f += 64) {
            uint32_t side, kk, c4;
            const floatx4 y = fetch(f, side, kk, c4);
            place(y, side, kk, c4);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores have been acknowledged
    };
    auto load_keys = [&](uint32_t kb) {
        const uint16_t *kblk = kplane + block_at(kb);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < kS; ++s)
                k[t][s] = *reinterpret_cast<const half8 *>(kblk + ((t * chunks + min(4u * s + g, chunks - 1)) * 16 + jl) * 8);
    };
    auto load_values = [&](uint32_t kb) {
        const uint16_t *vblk = vplane + block_at(kb);
#pragma unroll
        for (int c = 0; c < kTiles; ++c)
            v[c] = *reinterpret_cast<const half8 *>(vblk + min(16u * c + jl, D - 1) * kVBlock + 8 * g);
    };
    uint32_t kb = kb_begin + wave;
    if (kb < kb_end) append_rows(kb);
    {
        // (A wavefront without a block loads one and ignores it: behind a branch the wait for the queries
        // would be a wait for every load.)
        const uint32_t some = min(kb, (item.kv_len - 1) / kBlockKeys);
        load_keys(some);
        load_values(some);
    }
    __builtin_amdgcn_sched_barrier(0);

    // Q^T as three B operands: step s takes channels 8 (4s + g) .. + 7 of vector jl, times the power
    // of two that brings the vector's largest below 2^15; colscale takes it out of the scores again.
    half8 q[3][kS];
    float colscale;
    {
        float most = 0.0f;
#pragma unroll
        for (int s = 0; s < kS; ++s) {
            const bool has = 4u * s + g < chunks && jv < nvec;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[s][h][e] = has ? x[s][h][e] : 0.0f;
                    most = fmaxf(most, fabsf(x[s][h][e]));
                }
        }
        most = lanes4_max(most);
        const int up = 15 - __builtin_amdgcn_frexp_expf(most);  // (0 for zero and for what is not finite: 2^15)
        colscale = ldexpf(qscale, -up);
#pragma unroll
        for (int s = 0; s < kS; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                _Float16 h0, h1, h2;
                split3(ldexpf(x[s][e / 4][e % 4], up), h0, h1, h2);
                q[0][s][e] = h0, q[1][s][e] = h1, q[2][s][e] = h2;
            }
    }

    float m_run = -INFINITY, l_run = 0.0f;
    floatx4 o[kTiles];
#pragma unroll
    for (int c = 0; c < kTiles; ++c) o[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // What both walks do with a block's scores: cap, mask, running maximum and sum; sc becomes the
    // weights, and the return value what the earlier blocks' outputs are worth now.
    auto weigh = [&](uint32_t key0, float (&sc)[2][4]) -> float {
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t kp = key0 + 8 * g + 4 * t + r;
                float v = sc[t][r];
                if (softcap > 0.0f) v = softcap_log2(v, softcap, inv_cap);
                if (kp > colpos || kp < collo) v = -INFINITY;
                sc[t][r] = v;
                mx = fmaxf(mx, v);
            }
        mx = lanes4_max(mx);
        const float m_new = fmaxf(m_run, mx);
        const bool dead = m_new == -INFINITY;
        const float alpha = (dead || m_run == -INFINITY) ? (dead ? 1.0f : 0.0f) : fast_exp2(m_run - m_new);
        float sum = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (Nothing finite in sight so far: -inf weighs zero against a reference of zero,
                // and a NaN score stays NaN and takes the row with it.)
                const float pe = fast_exp2(sc[t][r] - (dead ? 0.0f : m_new) + kWeightShift);
                sc[t][r] = pe;
                sum += pe;
            }
        l_run = l_run * alpha + sum;
        m_run = m_new;
        return alpha;
    };

    for (; kb < kb_end; kb += W) {
        const uint32_t key0 = kb * kBlockKeys, next = kb + W;
        float sc[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                // (Only the last step can lie beyond head_dim, and then in half of the lanes.)
                if (s == kS - 1 && 4u * s + g >= chunks) k[t][s] = half8{};
#pragma unroll
                for (int h = 2; h >= 0; --h) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(k[t][s], q[h][s], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[t][r] = acc[r] * colscale;
        }
        if (next < kb_end) {
            append_rows(next);
            load_keys(next);
        }
        const float alpha = weigh(key0, sc);
        half8 w[3];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                _Float16 h0, h1, h2;
                split3(sc[t][r], h0, h1, h2);
                w[0][4 * t + r] = h0, w[1][4 * t + r] = h1, w[2][4 * t + r] = h2;
            }
        // A row no query of the tile sees may hold anything: kept out of P.V even as 0 * x.
        if (key0 + kBlockKeys > tile_hi || key0 < tile_lo) {
            const uint32_t first = key0 + 8 * g;
            const u32x4 keep = first_halves(tile_hi > first ? min(8u, tile_hi - first) : 0u) &
                               ~first_halves(tile_lo > first ? min(8u, tile_lo - first) : 0u);
#pragma unroll
            for (int c = 0; c < kTiles; ++c) v[c] = keep_halves(v[c], keep);
        }
#pragma unroll
        for (int c = 0; c < kTiles; ++c) {
            o[c] *= alpha;
#pragma unroll
            for (int h = 2; h >= 0; --h) o[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v[c], w[h], o[c], 0, 0, 0);
        }
        if (next < kb_end) load_values(next);
    }

    float all = l_run;
#pragma unroll
    for (int c = 0; c < kTiles; ++c) {
        all += (o[c][0] + o[c][1]) + (o[c][2] + o[c][3]);
        *reinterpret_cast<floatx4 *>(&sm_o[wave][c][lane][0]) = o[c];
    }
    // Sums that are not finite: again on the f32 pipe, an output tile at a time and the scores anew
    // for each, in rolled loops. The path is cold and small rather than fast.
    if (__builtin_amdgcn_ballot_w64(!(fabsf(all) < INFINITY)) != 0) {
#pragma unroll 1
        for (uint32_t c = 0; 16 * c < D; ++c) {
            m_run = -INFINITY;
            l_run = 0.0f;
            floatx4 out = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (uint32_t kb = kb_begin + wave; kb < kb_end; kb += W) {
                const uint32_t key0 = kb * kBlockKeys;
                const uint64_t at = uint64_t(ring_blocks ? kb % ring_blocks : kb) * (kVBlock * D);
                floatx4 acc[2] = {};
#pragma unroll 1
                for (uint32_t ch = g; ch < D; ch += 4) {  // head_dim is a multiple of 4: every lane takes each turn
                    const float qv = jv < nvec ? qp[ch] * qscale : 0.0f;
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            float(__builtin_bit_cast(_Float16, kplane[at + ((t * chunks + ch / 8) * 16 + jl) * 8 + ch % 8])), qv,
                            acc[t], 0, 0, 0);
                }
                float sc[2][4];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sc[t][r] = acc[t][r];
                out *= weigh(key0, sc);
                const half8 v = *reinterpret_cast<const half8 *>(vplane + at + (16 * c + jl) * kVBlock + 8 * g);
                // One product per query row of the tile, with the keys it does not see cleared: the
                // reference never reads those (crates/attention/src/attention.rs:160-173).
#pragma unroll 1
                for (uint32_t rr = row_first; rr <= row_last; ++rr) {
                    const uint32_t pos = min(item.pos0 + rr, item.kv_len - 1);
                    const uint32_t lo = lowest_visible(item.pos0 + rr, window, kv_lo);
                    floatx4 part = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const uint32_t kp = key0 + 8 * g + 4 * t + r;
                            const float x = kp <= pos && kp >= lo ? float(v[4 * t + r]) : 0.0f;
                            part = __builtin_amdgcn_mfma_f32_16x16x4f32(x, sc[t][r], part, 0, 0, 0);
                        }
                    if (row == rr) out += part;
                }
            }
            *reinterpret_cast<floatx4 *>(&sm_o[wave][c][lane][0]) = out;
        }
    }

    // ---- merge the wavefronts through LDS
    const float l_col = lanes4_sum(l_run);
    if (g == 0) {
        sm_m[wave][jl] = m_run;
        sm_l[wave][jl] = l_col;
    }
    __syncthreads();

    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, sm_m[w][jl]);
    float L = 0.0f, wgt[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const float mw = sm_m[w][jl];
        wgt[w] = mw == -INFINITY ? 0.0f : fast_exp2(mw - M);
        L = fmaf(sm_l[w][jl], wgt[w], L);
    }
    if (jv >= nvec) return;
    const bool final_out = item.splits == 1;
    const uint64_t ps = item.ws0 + (uint64_t(row) * p.q_heads + head) * item.splits + split;
    float *dst = final_out ? p.out + (uint64_t(item.q_row0 + row) * p.q_heads + head) * D : p.ws + ps * D;
    const float post = final_out ? 1.0f / L : 1.0f;
    // Tile c, lane (jl, g), register rr = channel 16c + 4g + rr: wavefront w finishes tiles w, w + 4, ..
    for (uint32_t c = wave; 16 * c < D; c += W) {
        floatx4 fin = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w) fin += *reinterpret_cast<const floatx4 *>(&sm_o[w][c][lane][0]) * wgt[w];
        fin *= post;
        *reinterpret_cast<floatx4 *>(dst + 16 * c + 4 * g) = fin;
    }
    if (!final_out && wave == 0 && g == 0)
        *reinterpret_cast<float2 *>(p.ws + uint64_t(total_partials) * D + ps * 2) = make_float2(M, L);
}

}  // namespace

bool attn_splitk_any_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows) {
    return g.head_dim % 4 == 0 && g.head_dim >= 4 && g.head_dim <= 256 && group >= 1 && max_rows >= 1;
}
// By the registers of a wavefront: up to 168, up to 256, and more than that.
uint32_t attn_splitk_any_groups_per_cu(const PoolGeom &g) {
    return g.head_dim <= 64 ? 3 : g.head_dim <= 128 ? 2 : 1;
}
// f32 steps bring their rows along (attn_splitk_rows_kernel.h: they are read where they are). So do
// f16 steps of up to 16 query vectors per KV head, and of a few rows more, of which every tile's workgroups
// that reach the new positions store all: 3 us of launch saved, a microsecond spent for eight rows
// (scattered stores of two bytes; head_dim 80, 32 Q / 8 KV heads, six rows at 450 12.5 -> 9.7 us a layer;
// twenty rows 9.9 -> 11.0). More than eight rows of wide heads are too many for the one wavefront that owns
// their block: head_dim 256, 8 Q / 8 KV heads, sixteen rows at 400 / 1,100 21.0 / 22.9 -> 15.6 / 16.7.
bool attn_splitk_any_appends(const PoolGeom &g, int elem_f16, uint32_t group, uint32_t max_rows) {
    return attn_splitk_any_supports(g, group, max_rows) && (!elem_f16 || max_rows <= 8 || (max_rows * group <= 16 && max_rows * g.head_dim <= 2048));
}

hipError_t launch_attn_splitk_any(int elem_f16, const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  hipStream_t stream) {
    if (b.total_blocks == 0) return hipSuccess;
    if (b.parts) return launch_attn_parts_halves(p, b, total_partials, stream);
    const uint32_t d = p.g.head_dim;
    // (Batches of one item take the eight-item argument block: 0.1 us on a launch of 5.)
#define ITAK_ANY(W, ...)                                                                          \
    do {                                                                                          \
        if (b.n <= 8) {                                                                           \
            constexpr int N = 8;                                                                  \
            launch_kernel(__VA_ARGS__, b.total_blocks, W * 64, 0, stream, p, AttnBatchT<N>(b), total_partials); \
        } else {                                                                                  \
            constexpr int N = 64;                                                                 \
            launch_kernel(__VA_ARGS__, b.total_blocks, W * 64, 0, stream, p, AttnBatchT<N>(b), total_partials); \
        }                                                                                         \
    } while (0)
#define ITAK_HALVES(DP)                                                        \
    do {                                                                       \
        if constexpr (DP <= 128) {                                             \
            if (b.on_eight) {                                                  \
                ITAK_ANY(8, attn_splitk_halves_kernel<DP, 8, N>);              \
                break;                                                         \
            }                                                                  \
        }                                                                      \
        ITAK_ANY(4, attn_splitk_halves_kernel<DP, 4, N>);                      \
    } while (0)
#define ITAK_ROWS(T, DP, TT)                                                   \
    do {                                                                       \
        if constexpr (DP <= 128) {                                             \
            if (b.on_eight) {                                                  \
                ITAK_ANY(8, attn_splitk_rows_kernel<T, DP, false, 1, false, 8, true, N>); \
                break;                                                         \
            }                                                                  \
        }                                                                      \
        if (b.half_blocks)                                                     \
            ITAK_ANY(4, attn_splitk_rows_kernel<T, DP, false, 1, false, 4, true, N>); \
        else                                                                   \
            ITAK_ANY(4, attn_splitk_rows_kernel<T, DP, false, TT, false, 4, false, N>); \
    } while (0)
    if (elem_f16 && p.g.v_block) {
        switch ((d + 31) / 32) {
            case 1: ITAK_HALVES(32); break;
            case 2: ITAK_HALVES(64); break;
            case 3: ITAK_HALVES(96); break;
            case 4: ITAK_HALVES(128); break;
            case 5: ITAK_HALVES(160); break;
            case 6: ITAK_HALVES(192); break;
            case 7: ITAK_HALVES(224); break;
            default: ITAK_HALVES(256); break;
        }
    } else if (elem_f16) {
        switch ((d + 63) / 64) {
            case 1: ITAK_ROWS(uint16_t, 64, 2); break;
            case 2: ITAK_ROWS(uint16_t, 128, 2); break;
            case 3: ITAK_ROWS(uint16_t, 192, 2); break;
            default: ITAK_ROWS(uint16_t, 256, 2); break;
        }
    } else {
        switch ((d + 63) / 64) {
            case 1: ITAK_ROWS(float, 64, 1); break;
            case 2: ITAK_ROWS(float, 128, 1); break;
            case 3: ITAK_ROWS(float, 192, 1); break;
            default: ITAK_ROWS(float, 256, 1); break;
        }
    }
#undef ITAK_ROWS
#undef ITAK_HALVES
#undef ITAK_ANY
    return hipGetLastError();
}

}  // namespace itak
