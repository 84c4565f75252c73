// Blocks of some rows (prompt chunks, longer speculative blocks) on f16 pools at head_dim 128,
// as tiles of 16 or 32 query vectors whose wavefronts share out the keys.
//
// One workgroup owns (item, KV head, tile, split of the context); a query vector is one query row of
// one Q head of the KV group, vectors counted densely (vector j = row j / group, head j % group).
// Each wavefront walks 32-key blocks of its own, newest first, K and V straight from their planes
// into MFMA operand registers, with a private online softmax; the wavefronts merge once through
// LDS. No synchronisation inside the walk.
//
// Against the block kernel (attn_prefill_f16_kernel.h), whose wavefronts share the keys and split
// the vectors: there a unit is 64 or 128 vectors, so a 61-row block over a window of 2,048 is 32 units that
// must be cut into eight runs of eight blocks to fill the device, each of which writes a partial of
// all its vectors (8 MB, and a merge launch that reads them). Here the same block is 124 units of
// 16 vectors whose eight wavefronts already are an eightfold split, merged in LDS: short contexts stay whole
// (no partials, no second launch), longer ones are cut in two or four. The price is that a tile reads the keys for
// 16 (32) vectors where the block kernel's ring feeds 64 (128): long walks are bound by the
// 64 bytes a clock that come into a compute unit through its vector cache, 16 KB in 0.11 us (`shared` below), so
// long contexts under many rows stay with the block kernel; the planner below weighs the two. Short ones are mostly what
// a launch takes whatever it walks (`fixed`, 5.4 to 7.3 us) and, split, the merge launch.
//
// New rows (AttnParams::k_new / v_new): the step's own keys and values are read where the caller left
// them, as f32 straight into the operand registers of the wavefronts whose first block holds them
// (at most one block each: a launch carries no more new blocks than a workgroup has
// wavefronts); workgroups of their own behind the others convert them once and store them to the
// planes. Nothing in the launch waits for those stores.
//
// Semantics: gqa_attention in crates/attention/src/attention.rs:104-215, softcap as
// crates/torch-math/src/logits.rs:26-37.
#include "attn_splitk_f16_kernel.h"

#include <math.h>

#include <algorithm>

namespace itak {

namespace {

constexpr uint32_t kTilesVectors = 4096;  // query vectors per KV head up to which (j * magic) >> 16 divides by the group
// How far scores may run ahead of a column's reference (log2). The block kernel's 8 keeps the rescaling of
// the accumulators off the common path (2.5 % of a step); steps the split-K kernel took keep its exact
// running maximum, since softmax weights round better in f16 just below a power of two, where the maximum puts the
// largest (error against 64 bits 2.5e-4 with 0, 2.8e-4 with 8).
constexpr float kTileSlack = 8.0f;

// K/V are read once per tile: the next tile finds them in L2, so they are asked for without the
// streaming hint (61 rows over a window of 2,048 left whole, with an append launch: 21.8 -> 20.3 us; from 30 blocks
// per compute unit on, where tiles no longer meet in L2, the hint would be the better choice, and other kernels are).
__device__ __forceinline__ void tile_load_keys(BlockOperands &b, const uint16_t *kplane, uint32_t sb, uint32_t g,
                                               uint32_t i) {
    const uint16_t *base = kplane + uint64_t(sb) * (kBlockKeys * kD) + (g * 16 + i) * 8;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            b.k[t][s] = *reinterpret_cast<const half8 *>(base + ((t * 16 + s * 4) * 16) * 8);
}
__device__ __forceinline__ void tile_load_values(BlockOperands &b, const uint16_t *vplane, uint32_t sb, uint32_t g,
                                                 uint32_t i) {
    const uint16_t *base = vplane + uint64_t(sb) * (kBlockKeys * kD) + i * kBlockKeys + g * 8;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) b.v[dt] = *reinterpret_cast<const half8 *>(base + dt * 16 * kBlockKeys);
}

// The operand elements of keys [pos0, end) of block kb, from the caller's f32 rows (kn, vn: row 0 =
// position pos0, this KV head's channels). A NaN keeps its own payload here, where the planes
// hold the canonical one: as an operand it is a NaN either way.
__device__ __forceinline__ void tile_take_new(BlockOperands &b, const float *kn, const float *vn, uint32_t row_width,
                                              uint32_t kb, uint32_t g, uint32_t i, uint32_t pos0, uint32_t end) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t key = kb * kBlockKeys + (i >> 2) * 8 + t * 4 + (i & 3);
        const bool is_new = key >= pos0 && key < end;
        const float *src = kn + uint64_t(is_new ? key - pos0 : 0) * row_width + g * 8;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const floatx4 a = *reinterpret_cast<const floatx4 *>(src + s * 32);
            const floatx4 c = *reinterpret_cast<const floatx4 *>(src + s * 32 + 4);
            const half8 h{static_cast<_Float16>(a[0]), static_cast<_Float16>(a[1]), static_cast<_Float16>(a[2]),
                          static_cast<_Float16>(a[3]), static_cast<_Float16>(c[0]), static_cast<_Float16>(c[1]),
                          static_cast<_Float16>(c[2]), static_cast<_Float16>(c[3])};
            const u32x4 hb = __builtin_bit_cast(u32x4, h), kbits = __builtin_bit_cast(u32x4, b.k[t][s]);
            u32x4 r;
#pragma unroll
            for (int x = 0; x < 4; ++x) r[x] = is_new ? hb[x] : kbits[x];
            b.k[t][s] = __builtin_bit_cast(half8, r);
        }
    }
    const uint32_t key_base = kb * kBlockKeys + g * 8;
    const uint32_t n_end = min(end - min(end, key_base), 8u), n_first = min(pos0 - min(pos0, key_base), 8u);
    const u32x4 take = first_halves(n_end) & ~first_halves(n_first);
    // (Keys that are not new read a row that is there.)
    const uint32_t rows = end - pos0;
    uint32_t at[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t r = key_base + e - pos0;
        at[e] = (r < rows ? r : 0) * row_width + i;
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
        half8 h;
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = static_cast<_Float16>(vn[at[e] + dt * 16]);
        b.v[dt] = __builtin_bit_cast(half8, (__builtin_bit_cast(u32x4, b.v[dt]) & ~take) |
                                                (__builtin_bit_cast(u32x4, h) & take));
    }
}

// One 32-key block's new rows of one KV head, converted and stored to the planes by four wavefronts: two take the
// values, eight keys of four channels a lane, two the keys, eight channels of four rows a lane, every load issued
// before the first is waited for. A workgroup stores up to kStoreTurns blocks for every four wavefronts it has, one
// after the other beside the walks of the others: with a workgroup a block, 61 rows on 2,040 positions were 248 tiles
// and 12 of these on 256 compute units that hold one each, and some ran a second round:
// 15.4 -> 14.5 us a layer (with a window of 2,048 around them 16.2 -> 15.8); 20 rows on 500 of four slots 9.4 -> 8.9,
// 61 rows on none 6.3 -> 6.1, 500 on none 15.1 -> 14.7.
constexpr uint32_t kStoreTurns = 2;
__device__ __forceinline__ void tile_store_new(const AttnParams &p, const AttnItem &item, uint32_t kv_head, uint32_t kb,
                                               uint16_t *kplane, uint16_t *vplane) {
    const uint32_t tid = threadIdx.x & 255;
    const uint32_t row_width = p.g.kv_heads * kD;
    const uint32_t sb = p.ring_blocks ? kb % p.ring_blocks : kb;
    const uint32_t first = kb * kBlockKeys - item.pos0, rows = item.rows;  // row of the block's first key (may wrap)
    const uint32_t lane = tid & 127;
    const uint64_t at = uint64_t(item.q_row0) * row_width + kv_head * kD;
    floatx4 x[8];
    if (tid < 128) {  // values: keys 8 * eight .., channels 4 * c ..
        const uint32_t eight = lane >> 5, c = (lane & 31) * 4;
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) {
            const uint32_t r = first + eight * 8 + e;
            x[e] = *reinterpret_cast<const floatx4 *>(p.v_new + at + uint64_t(r < rows ? r : 0) * row_width + c);
        }
        uint32_t there = 0;
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) there |= first + eight * 8 + e < rows ? 1u << e : 0u;
        uint16_t *dst = vplane + uint64_t(sb) * (kBlockKeys * kD) + c * kBlockKeys + eight * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint16_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = f32_to_f16_bits(x[e][j]);
            if (there == 0xffu) {
                uint4 w;
                w.x = h[0] | uint32_t(h[1]) << 16, w.y = h[2] | uint32_t(h[3]) << 16;
                w.z = h[4] | uint32_t(h[5]) << 16, w.w = h[6] | uint32_t(h[7]) << 16;
                *reinterpret_cast<uint4 *>(dst + j * kBlockKeys) = w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (there >> e & 1u) dst[j * kBlockKeys + e] = h[e];
            }
        }
    } else {  // keys: channels 8 * chunk .. of rows kin, kin + 8, ..
        const uint32_t chunk = lane & 15;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t r = first + (lane >> 4) + 8 * u;
            const float *src = p.k_new + at + uint64_t(r < rows ? r : 0) * row_width + chunk * 8;
            x[2 * u] = *reinterpret_cast<const floatx4 *>(src), x[2 * u + 1] = *reinterpret_cast<const floatx4 *>(src + 4);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t kin = (lane >> 4) + 8 * u, kt = (kin >> 2) & 1, ki = (kin >> 3) * 4 + (kin & 3);
            uint16_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = f32_to_f16_bits(x[2 * u + (e >> 2)][e & 3]);
            uint4 w;
            w.x = h[0] | uint32_t(h[1]) << 16, w.y = h[2] | uint32_t(h[3]) << 16;
            w.z = h[4] | uint32_t(h[5]) << 16, w.w = h[6] | uint32_t(h[7]) << 16;
            if (first + kin < rows)
                *reinterpret_cast<uint4 *>(kplane + uint64_t(sb) * (kBlockKeys * kD) + ((kt * 16 + chunk) * 16 + ki) * 8) = w;
        }
    }
}

constexpr size_t tiles_lds(int nq, int waves) {
    return (size_t(2) * waves * nq * 16 + size_t(waves) * nq * 8 * 64 * 4) * 4 + size_t(nq) * 16 * kQStride * 2;
}

struct TilesExtra {
    const float *gate;    // the output is multiplied by sigmoid(gate) where this launch writes it, or null
    uint32_t stores;      // workgroups that store an item's new rows, a KV head (0: nothing to append)
    float slack;
};

template <int NQ, int WAVES, int N, bool RING>
__global__ __launch_bounds__(WAVES * 64, NQ == 1 && WAVES == 4 ? 3 : 2) void attn_tiles_f16_kernel(AttnParams p, AttnBatchT<N> b, uint32_t total_partials,
                                                                    TilesExtra extra) {
    extern __shared__ float lds[];
    float *sm_m = lds;                     // [WAVES][NQ*16]
    float *sm_l = sm_m + WAVES * NQ * 16;  // [WAVES][NQ*16]
    float *sm_o = sm_l + WAVES * NQ * 16;  // [WAVES][NQ][8][64][4]
    _Float16 *sm_q = reinterpret_cast<_Float16 *>(sm_o + WAVES * NQ * 8 * 64 * 4);  // [NQ*16][kQStride]
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t g = lane >> 4, jl = lane & 15;

    // (Every argument in one batch of scalar loads, see attn_splitk_f16_body.)
    if (N == 1)
        asm volatile("" ::"s"(p.layer_base), "s"(p.q), "s"(p.out), "s"(p.ws), "s"(p.k_new), "s"(p.v_new),
                     "s"(p.g.slot_stride), "s"(p.g.head_stride), "s"(p.g.side_stride), "s"(p.g.kv_heads), "s"(p.q_heads),
                     "s"(p.group), "s"(p.group_magic), "s"(p.scale), "s"(p.softcap), "s"(total_partials),
                     "s"(b.total_blocks), "s"(b.item[0].slot), "s"(b.item[0].rows), "s"(b.item[0].pos0),
                     "s"(b.item[0].q_row0), "s"(b.item[0].kv_len), "s"(b.item[0].splits), "s"(b.item[0].keys_per_split),
                     "s"(b.item[0].block0), "s"(b.item[0].ws0), "s"(b.item[0].splits_magic), "s"(b.item[0].kv_lo),
                     "s"(p.window), "s"(p.ring_blocks), "s"(extra.gate), "s"(extra.stores), "s"(extra.slack));
    const uint32_t group = p.group, magic = p.group_magic, kv_heads = p.g.kv_heads;
    if (blockIdx.x >= b.total_blocks) {  // (item, KV head, some blocks) of the new rows, to the planes
        const uint32_t at = blockIdx.x - b.total_blocks, unit = at / extra.stores;
        const AttnItem item = b.item[N == 1 ? 0 : unit / kv_heads];
        const uint32_t kv_head = unit % kv_heads;
        uint16_t *kplane = static_cast<uint16_t *>(const_cast<void *>(p.layer_base)) + item.slot * p.g.slot_stride +
                           kv_head * p.g.head_stride;
        uint32_t kb = item.pos0 / kBlockKeys + (at - unit * extra.stores) * (WAVES / 4) * kStoreTurns + tid / 256;
#pragma unroll 1
        for (uint32_t turn = 0; turn < kStoreTurns && kb * kBlockKeys < item.pos0 + item.rows; ++turn, kb += WAVES / 4)
            tile_store_new(p, item, kv_head, kb, kplane, kplane + p.g.side_stride);
        return;
    }
    const AttnItem item = b.of_block(blockIdx.x);
    const uint32_t nvec = item.rows * group;
    // Eight units (KV head, split) after eight others, and within the eight a tile after the other:
    // workgroup i runs on compute die i mod 8, so the tiles of a unit, which read the same keys and
    // values, find them in one L2. The last tile, which sees the most, first.
    constexpr uint32_t kVec = NQ * 16;
    uint32_t local = blockIdx.x - item.block0;
    const uint32_t tiles = (nvec + kVec - 1) / kVec, units = kv_heads * item.splits;
    const uint32_t eight = local / (8 * tiles), in = local - eight * 8 * tiles;
    const uint32_t held = min(8u, units - eight * 8);
    const uint32_t tile = in / held;
    local = eight * 8 + in - tile * held;
    const uint32_t vec0 = (tiles - 1 - tile) * kVec;
    const uint32_t kv_head = item.splits > 1 ? __umulhi(local, item.splits_magic) : local;
    const uint32_t split = local - kv_head * item.splits;
    const uint32_t row_first = (vec0 * magic) >> 16, row_last = (min(vec0 + kVec - 1, nvec - 1) * magic) >> 16;

    const uint16_t *kplane =
        static_cast<const uint16_t *>(p.layer_base) + item.slot * p.g.slot_stride + kv_head * p.g.head_stride;
    const uint16_t *vplane = kplane + p.g.side_stride;
    const uint32_t row_width = kv_heads * kD;

    // What the tile's rows see: positions [lo_min, seen_end); its blocks of the split's run.
    const uint32_t ring_blocks = RING ? p.ring_blocks : 0;
    const uint32_t window = RING ? p.window : 0, kv_lo = RING ? item.kv_lo : 0;
    const uint32_t lo_min = lowest_visible(item.pos0 + row_first, window, kv_lo);
    const uint32_t lo_max = lowest_visible(item.pos0 + row_last, window, kv_lo);
    const uint32_t first_pos = min(item.pos0 + row_first, item.kv_len - 1);
    const uint32_t seen_end = min(item.pos0 + row_last + 1, item.kv_len);
    const uint32_t run0 = (RING ? item_first_block(item) : 0) + split * (item.keys_per_split / kBlockKeys);
    const uint32_t kb_begin = RING ? max(run0, lo_min / kBlockKeys) : run0;
    const uint32_t kb_end = min((seen_end + kBlockKeys - 1) / kBlockKeys, run0 + item.keys_per_split / kBlockKeys);
    const bool fused = p.k_new != nullptr;

    // ---- the query vectors (padding vectors re-read the last real one and are zeroed when staged)
    constexpr int QL = (NQ * 16 * (kD / 4)) / (WAVES * 64);
    static_assert(QL >= 1, "too many wavefronts for the query tile");
    float4 qld[QL];
#pragma unroll
    for (int u = 0; u < QL; ++u) {
        const uint32_t f = tid + u * WAVES * 64;
        const uint32_t j = min(vec0 + (f >> 5), nvec - 1), c4 = (f & 31) * 4;
        const uint32_t row = (j * magic) >> 16, head = kv_head * group + (j - row * group);
        qld[u] = *reinterpret_cast<const float4 *>(p.q + (uint64_t(item.q_row0 + row) * p.q_heads + head) * kD + c4);
    }

    // ---- the wavefront's first block, the newest it has (one without any loads the run's first)
    int32_t kb = int32_t(kb_end) - 1 - int32_t(wave);
    const bool has_block = kb >= int32_t(kb_begin);
    BlockOperands buf;
    uint32_t sb = storage_block(has_block ? uint32_t(kb) : run0, ring_blocks);
    tile_load_keys(buf, kplane, sb, g, jl);
    tile_load_values(buf, vplane, sb, g, jl);

    uint32_t colpos[NQ], collo[NQ];
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt) {
        const uint32_t row = ((vec0 + qt * 16 + jl) * magic) >> 16;
        colpos[qt] = min(item.pos0 + row, item.kv_len - 1);
        collo[qt] = lowest_visible(item.pos0 + row, window, kv_lo);
    }
    const float softcap = p.softcap, slack = extra.slack;
    // With a softcap the scores come out as the argument of tanh's exponential (2 log2(e) s / cap).
    const float cap2 = softcap * kLog2e;
    const float qscale = softcap > 0.0f ? p.scale * (2.0f * kLog2e / softcap) : p.scale * kLog2e;
#pragma unroll
    for (int u = 0; u < QL; ++u) {
        const uint32_t f = tid + u * WAVES * 64;
        const uint32_t j = f >> 5, c4 = (f & 31) * 4;
        half4 h{static_cast<_Float16>(qld[u].x * qscale), static_cast<_Float16>(qld[u].y * qscale),
                static_cast<_Float16>(qld[u].z * qscale), static_cast<_Float16>(qld[u].w * qscale)};
        if (vec0 + j >= nvec) h = half4{0, 0, 0, 0};
        *reinterpret_cast<half4 *>(sm_q + j * kQStride + c4) = h;
    }
    __syncthreads();
    half8 qreg[NQ][4];
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            qreg[qt][k] = *reinterpret_cast<const half8 *>(sm_q + (qt * 16 + jl) * kQStride + k * 32 + g * 8);
    if (fused && has_block && (uint32_t(kb) + 1) * kBlockKeys > item.pos0) {
        const uint64_t at = uint64_t(item.q_row0) * row_width + kv_head * kD;
        tile_take_new(buf, p.k_new + at, p.v_new + at, row_width, uint32_t(kb), g, jl, item.pos0, seen_end);
    }

    // ---- the walk. The softmax's reference per column, its threshold and the denominator through
    // the matrix pipe are the block kernel's: the reference is the accumulators' start and
    // moves only when a score runs more than `slack` ahead of it. One set of operand registers:
    // the next block's keys are asked for when the scores have used this one's, its values when the
    // products have.
    const half8 ones = {_Float16(1.0f), _Float16(1.0f), _Float16(1.0f), _Float16(1.0f),
                        _Float16(1.0f), _Float16(1.0f), _Float16(1.0f), _Float16(1.0f)};
    float ref[NQ], thr[NQ];
    floatx4 l[NQ], o[NQ][8];
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt) {
        ref[qt] = 0.0f;
        thr[qt] = -INFINITY;
        l[qt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[qt][dt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const RowSpan span{item.pos0, row_first, row_last + 1, vec0, window, kv_lo, magic, false, false};
    for (; kb >= int32_t(kb_begin); kb -= WAVES) {
        const uint32_t base = uint32_t(kb) * kBlockKeys, key_base = base + g * 8;
        const bool more = kb - WAVES >= int32_t(kb_begin);
        if (more) sb = !RING || sb >= WAVES ? sb - WAVES : storage_block(uint32_t(kb - WAVES), ring_blocks);
        floatx4 x[NQ][2];
#pragma unroll
        for (int qt = 0; qt < NQ; ++qt)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float nr = softcap > 0.0f ? 0.0f : -ref[qt];
                floatx4 s = floatx4{nr, nr, nr, nr};
#pragma unroll
                for (int k = 0; k < 4; ++k) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(buf.k[t][k], qreg[qt][k], s, 0, 0, 0);
                x[qt][t] = s;
            }
        if (more) tile_load_keys(buf, kplane, sb, g, jl);
        if (softcap > 0.0f) {
#pragma unroll
            for (int qt = 0; qt < NQ; ++qt)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[qt][e >> 2][e & 3] = softcap_of_exp2_arg(x[qt][e >> 2][e & 3], cap2, ref[qt]);
        }
        const bool need_mask = base + kBlockKeys > first_pos + 1 || (RING && base < lo_max);
        if (need_mask) {
#pragma unroll
            for (int qt = 0; qt < NQ; ++qt)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (key_base + e > colpos[qt] || (RING && key_base + e < collo[qt])) x[qt][e >> 2][e & 3] = -INFINITY;
        }
        float lmax[NQ];
        bool over = false;
#pragma unroll
        for (int qt = 0; qt < NQ; ++qt) {
            float mx = max3(x[qt][0][0], x[qt][0][1], x[qt][0][2]);
            mx = max3(mx, x[qt][0][3], x[qt][1][0]);
            mx = max3(mx, x[qt][1][1], x[qt][1][2]);
            lmax[qt] = max3(mx, x[qt][1][3], x[qt][1][3]);
            over = over || lmax[qt] > thr[qt];
        }
        if (__builtin_amdgcn_ballot_w64(over) != 0) {
#pragma unroll
            for (int qt = 0; qt < NQ; ++qt) {
                const float cm = column_max(lmax[qt]);
                const bool live = thr[qt] != -INFINITY;
                float delta = live ? fmaxf(cm, 0.0f) : cm;
                if (cm == -INFINITY) delta = 0.0f;
                const float alpha = live ? fast_exp2(-delta) : 1.0f;
                ref[qt] += delta;
                if (cm != -INFINITY) thr[qt] = slack;
                l[qt] *= alpha;
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) o[qt][dt] *= alpha;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[qt][t][r] -= delta;
            }
        }
        half8 pb[NQ];
#pragma unroll
        for (int qt = 0; qt < NQ; ++qt) {
#pragma unroll
            for (int e = 0; e < 8; ++e) pb[qt][e] = static_cast<_Float16>(fast_exp2(x[qt][e >> 2][e & 3]));
        }
        if (need_mask) {
            // Rows that no row of the tile sees (stale, not stored yet, or other tiles') stay out of P.V
            // even as 0 * x; a value that is not finite in a key that only some rows see goes the exact
            // way (accumulate_by_row).
            const uint32_t end = min(seen_end - min(seen_end, key_base), 8u);
            const uint32_t first = RING ? min(lo_min - min(lo_min, key_base), 8u) : 0u;
            const u32x4 keep = first_halves(end) & ~first_halves(first);
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) buf.v[dt] = keep_halves(buf.v[dt], keep);
            if (row_last > row_first && __builtin_expect(any_not_finite(buf.v), false)) {
#pragma unroll
                for (int qt = 0; qt < NQ; ++qt)
                    accumulate_by_row<RING>(o[qt], buf, pb[qt], qt, key_base, jl, seen_end, span);
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) buf.v[dt] = half8{0, 0, 0, 0, 0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int qt = 0; qt < NQ; ++qt) {
            l[qt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pb[qt], l[qt], 0, 0, 0);
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
                o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(buf.v[dt], pb[qt], o[qt][dt], 0, 0, 0);
        }
        if (more) tile_load_values(buf, vplane, sb, g, jl);
    }

    // ---- merge the wavefronts through LDS; every read is issued before the first is used
    constexpr int kDtPerWave = 8 / WAVES;  // channel tiles each wavefront finishes
    const bool final_out = item.splits == 1;
    const bool gated = final_out && extra.gate != nullptr;
    uint32_t jl_again = jl;  // (worked out again here: kept from the prologue they would hold registers)
    asm volatile("" : "+v"(jl_again));
    uint32_t colout[NQ], colps[NQ];
    float4 gt[NQ][kDtPerWave];
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt) {
        const uint32_t j = min(vec0 + qt * 16 + jl_again, nvec - 1);
        const uint32_t row = (j * magic) >> 16, head = kv_head * group + (j - row * group);
        colout[qt] = (item.q_row0 + row) * p.q_heads + head;
        colps[qt] = item.ws0 + (row * p.q_heads + head) * item.splits + split;
        if (gated) {
#pragma unroll
            for (int c = 0; c < kDtPerWave; ++c)
                gt[qt][c] = *reinterpret_cast<const float4 *>(extra.gate + uint64_t(colout[qt]) * kD +
                                                              (wave * kDtPerWave + c) * 16 + g * 4);
        }
    }
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt) {
        if (g == 0) {
            sm_m[wave * NQ * 16 + qt * 16 + jl] = thr[qt] == -INFINITY ? -INFINITY : ref[qt];
            sm_l[wave * NQ * 16 + qt * 16 + jl] = l[qt][0];
        }
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
            *reinterpret_cast<floatx4 *>(sm_o + (((wave * NQ + qt) * 8 + dt) * 64 + lane) * 4) = o[qt][dt];
    }
    __syncthreads();
    float *const ws_acc = p.ws;
    float *const ws_ml = p.ws + uint64_t(total_partials) * kD;
#pragma unroll
    for (int qt = 0; qt < NQ; ++qt) {
        floatx4 ow[kDtPerWave][WAVES];
        float mw[WAVES], lw[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            mw[w] = sm_m[w * NQ * 16 + qt * 16 + jl];
            lw[w] = sm_l[w * NQ * 16 + qt * 16 + jl];
        }
#pragma unroll
        for (int c = 0; c < kDtPerWave; ++c)
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
                ow[c][w] = *reinterpret_cast<const floatx4 *>(
                    sm_o + (((w * NQ + qt) * 8 + wave * kDtPerWave + c) * 64 + lane) * 4);
        float M = mw[0];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) M = fmaxf(M, mw[w]);
        float L = 0.0f, wgt[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            wgt[w] = mw[w] == -INFINITY ? 0.0f : fast_exp2(mw[w] - M);
            L = fmaf(lw[w], wgt[w], L);
        }
        if (vec0 + qt * 16 + jl >= nvec) continue;
        float *dst = final_out ? p.out + uint64_t(colout[qt]) * kD : ws_acc + uint64_t(colps[qt]) * kD;
        const float post = final_out ? 1.0f / L : 1.0f;
#pragma unroll
        for (int c = 0; c < kDtPerWave; ++c) {
            floatx4 acc = ow[c][0] * wgt[0];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) acc += ow[c][w] * wgt[w];
            acc *= post;
            if (gated)
                acc = floatx4{acc[0] * sigmoid_fast(gt[qt][c].x), acc[1] * sigmoid_fast(gt[qt][c].y),
                              acc[2] * sigmoid_fast(gt[qt][c].z), acc[3] * sigmoid_fast(gt[qt][c].w)};
            *reinterpret_cast<floatx4 *>(dst + (wave * kDtPerWave + c) * 16 + g * 4) = acc;
        }
        if (!final_out && wave == 0 && g == 0)
            *reinterpret_cast<float2 *>(ws_ml + uint64_t(colps[qt]) * 2) = make_float2(M, L);
    }
}

template <int NQ, int WAVES, int N, bool RING>
hipError_t launch_tiles(const AttnParams &p, const AttnBatch &b, uint32_t total_partials, const TilesExtra &extra,
                        hipStream_t stream) {
    constexpr size_t lds = tiles_lds(NQ, WAVES);
    static const hipError_t granted =
        hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_tiles_f16_kernel<NQ, WAVES, N, RING>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (granted != hipSuccess) return granted;
    launch_kernel(attn_tiles_f16_kernel<NQ, WAVES, N, RING>, b.total_blocks + b.n * p.g.kv_heads * extra.stores,
                  WAVES * 64, lds, stream, p, AttnBatchT<N>(b), total_partials, extra);
    return hipGetLastError();
}

}  // namespace

bool attn_tiles_f16_supports(const PoolGeom &g, uint32_t group, uint32_t most_rows) {
    return g.v_block == kVBlock && g.head_dim == kD && group >= 1 && group <= 16 && most_rows * group <= kTilesVectors;
}

// Fills splits / keys_per_split / block0 / ws0 for a batch in runs of at most `run` blocks.
static uint32_t fill_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, uint32_t nq, uint32_t run) {
    const uint32_t group = q_heads / g.kv_heads;
    uint32_t block0 = 0, ws0 = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        AttnItem &it = b.item[i];
        const uint32_t blocks = item_block_count(it);
        const uint32_t splits = std::max((blocks + run - 1) / run, 1u);
        const uint32_t each = std::max((blocks + splits - 1) / splits, 1u);
        it.splits = std::max((blocks + each - 1) / each, 1u);
        it.keys_per_split = each * kBlockKeys;
        it.splits_magic = it.splits > 1 ? uint32_t(((uint64_t(1) << 32) + it.splits - 1) / it.splits) : 0;
        it.block0 = block0;
        it.ws0 = ws0;
        block0 += g.kv_heads * ((it.rows * group + nq * 16 - 1) / (nq * 16)) * it.splits;
        if (it.splits > 1) ws0 += it.rows * q_heads * it.splits;
    }
    b.total_blocks = block0;
    b.rows_per_block = 0;
    return ws0;
}

// What a form costs in microseconds, a launch's gap included: `fixed`, its walk, and with several splits
// the merge launch and the partials' bytes. `alone` is a block's time where a workgroup has its compute
// unit to itself, `shared` what a block of every further workgroup there adds. The figures are a fit to
// 780 shapes (9 to 1,024 rows on 0 to 12,000 positions, 2 to 8 rows of 1 to 8 slots on 100 to 8,192, windows of 512
// and 2,048, five head layouts, as many layers as the last-level cache does not hold; every form and up
// to thirteen counts of splits timed for each): 6 % off on average, the pick 0.8 % behind the best. Both figures are of the
// launches as they were timed. Since then the merge launch asks for the partials there are (0.3 to 0.8 us less) and a
// chunk's rows are stored by fewer workgroups (0.2 to 0.9 us less), the same in each form: splits and these forms are priced a
// little too high, which costs steps near a line and no others.
struct TileForm {
    uint32_t sets, waves, resident;  // resident: workgroups a compute unit holds
    float fixed, alone, shared;
};
constexpr TileForm kForms[] = {
    {1, 4, 3, 5.43f, 0.165f, 0.112f}, {1, 8, 1, 6.17f, 0.137f, 0.114f},
    {2, 4, 2, 6.46f, 0.197f, 0.098f}, {2, 8, 1, 7.32f, 0.151f, 0.137f}};
constexpr float kBeside = 1.04f;                              // a walk's own blocks beside another workgroup's
constexpr float kMergeLaunch = 2.43f, kMergeRate = 1.71e6f;   // us, bytes a us
constexpr float kReadRate = 12.8e6f;                          // K/V once, what of it shows
constexpr float kRound = 2.65f;                               // each further round of resident workgroups
constexpr float kAppendLaunch = 2.6f, kAppendRow = 0.007f;    // a launch of its own for the new rows

// Most blocks that hold new rows, over the items.
static uint32_t most_new_blocks(const AttnBatch &b) {
    uint32_t most = 0;
    for (uint32_t i = 0; i < b.n; ++i)
        most = std::max(most, (b.item[i].pos0 + b.item[i].rows - 1) / kBlockKeys - b.item[i].pos0 / kBlockKeys + 1);
    return most;
}

// What a form walks, whatever the split: an item's blocks, its tiles over all KV heads, and what one of them sees.
struct TileItem {
    uint32_t blocks, units;
    float seen;
};
struct TileWork {
    TileItem item[kMaxBatchItems];
    uint64_t groups = 0, read = 0;  // workgroups of the whole contexts; bytes of keys and values, once
    float total = 0.0f;             // blocks that all workgroups see
};
static void work_of(const PoolGeom &g, const AttnBatch &b, uint32_t group, uint32_t window, const TileForm &f, TileWork &w) {
    const uint32_t vectors = f.sets * 16;
    for (uint32_t i = 0; i < b.n; ++i) {
        const AttnItem &it = b.item[i];
        const uint32_t blocks = item_block_count(it), tiles = (it.rows * group + vectors - 1) / vectors;
        const uint32_t units = g.kv_heads * tiles;
        // What a tile sees of them: its rows' window, or on average half the new rows less.
        const float seen = window ? float(std::min(blocks, (window + vectors / group + 62) / kBlockKeys))
                                  : std::max(float(blocks) - (tiles > 1 ? float(it.rows) / 64.0f : 0.0f), 1.0f);
        w.item[i] = {blocks, units, seen};
        w.groups += units;
        w.total += float(units) * seen;
        w.read += uint64_t(g.kv_heads) * blocks * 2 * kBlockKeys * kD * 2;
    }
}
// No split of the form takes less: its launch, what it reads, and the walks that share compute units.
static float least_of(const TileForm &f, const TileWork &w, uint64_t cus) {
    const float beside = w.groups > cus ? w.total * f.shared * (1.0f / float(cus) - 1.0f / float(w.groups)) : 0.0f;
    return (f.fixed + float(w.read) / kReadRate + beside) * 0.9999f;  // (sums in another order than cost_of's)
}
static float cost_of(const AttnBatch &b, uint32_t q_heads, const TileForm &f, const TileWork &w, uint32_t run, uint64_t cus,
                     uint64_t *partial_bytes) {
    uint64_t groups = 0, partials = 0;
    float longest = 0.0f;
    for (uint32_t i = 0; i < b.n; ++i) {
        const TileItem &it = w.item[i];
        const uint32_t splits = std::max((it.blocks + run - 1) / run, 1u);
        groups += uint64_t(it.units) * splits;
        longest = std::max(longest, std::min(float((it.blocks + splits - 1) / splits), it.seen));
        if (splits > 1) partials += uint64_t(b.item[i].rows) * q_heads * splits;
    }
    float walk = longest * f.alone;
    const uint64_t each_cu = (groups + cus - 1) / cus;
    if (each_cu > 1) walk = kBeside * walk + float(each_cu - 1) * w.total / float(groups) * f.shared;
    walk += float(w.read) / kReadRate;
    const uint64_t held = cus * f.resident;
    *partial_bytes = partials * (kD + 2) * 4;
    return f.fixed + walk + float((groups + held - 1) / held - 1) * kRound +
           (partials ? kMergeLaunch + float(*partial_bytes) / kMergeRate : 0.0f);
}

// (Forms that cannot come under the least so far, or under `below`, are not searched: 32 slots of nine rows at 1,000, which
// stay with the block kernel: 11.9 us of planning on one host core with the search unbounded and that kernel planned
// twice, 6.5 so.)
float attn_tiles_f16_choose(const PoolGeom &g, const AttnBatch &b, uint32_t q_heads, uint32_t window, bool brings_rows,
                            bool few_rows, uint64_t partial_limit, float below, TilesPlan &plan) {
    const uint64_t cus = compute_units();
    const uint32_t group = q_heads / g.kv_heads;
    uint32_t most = 1, rows = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        most = std::max(most, item_block_count(b.item[i]));
        rows += b.item[i].rows;
    }
    const uint32_t new_blocks = brings_rows ? most_new_blocks(b) : 0;
    constexpr uint8_t kCounts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32};
    float least = below;
    for (const TileForm &f : kForms) {
        if (f.sets == 2 && b.n == 1 && b.item[0].rows * group <= 16) continue;
        // (A wavefront takes at most one block of new rows.)
        const bool appends = new_blocks <= f.waves;
        const float append = appends ? 0.0f : kAppendLaunch + kAppendRow * float(rows);
        TileWork w;
        work_of(g, b, group, window, f, w);
        if (append + least_of(f, w, cus) >= least) continue;
        uint32_t before = 0;
        for (uint32_t c = 0; c < sizeof(kCounts); c += b.n > 8 ? 2 : 1) {
            const uint32_t run = (most + kCounts[c] - 1) / kCounts[c];
            if (run == before) continue;
            if (c && run * 2 < f.waves) break;
            before = run;
            // (The split-K kernel's whole steps have eight wavefronts: no more blocks under one maximum here.)
            if (few_rows && run > (f.waves == 4 ? 4u : g.kv_heads >= 8 ? 8u : 16u)) continue;
            if (few_rows && run < most && b.n > 1) break;
            uint64_t partial_bytes = 0;
            const float cost = append + cost_of(b, q_heads, f, w, run, cus, &partial_bytes);
            if (partial_limit && partial_bytes > partial_limit) break;
            if (cost < least) {
                least = cost;
                plan = TilesPlan{f.sets, f.waves, run, brings_rows && appends, few_rows};
            }
        }
    }
    return least;
}

uint32_t attn_tiles_f16_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, const TilesPlan &plan) {
    b.tile_sets = plan.sets;
    b.tile_waves = plan.waves;
    b.tile_exact = plan.exact ? 1 : 0;
    return fill_plan(g, b, q_heads, plan.sets, plan.run);
}

hipError_t launch_attn_tiles_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials, const float *gate,
                                 hipStream_t stream) {
    if (b.total_blocks == 0) return hipSuccess;
    const uint32_t new_blocks = p.k_new ? most_new_blocks(b) : 0, stored = b.tile_waves / 4 * kStoreTurns;
    if (new_blocks > b.tile_waves) return hipErrorInvalidValue;  // (the planner brings no more)
    const TilesExtra extra{gate, (new_blocks + stored - 1) / stored, b.tile_exact ? 0.0f : kTileSlack};
    hipError_t e = hipSuccess;
#define ITAK_TILES(NQ, W)                                                                          \
    do {                                                                                           \
        if (p.ring_blocks)                                                                         \
            ITAK_DISPATCH_BATCH(b.n, (e = launch_tiles<NQ, W, N, true>(p, b, total_partials, extra, stream)));  \
        else                                                                                       \
            ITAK_DISPATCH_BATCH(b.n, (e = launch_tiles<NQ, W, N, false>(p, b, total_partials, extra, stream))); \
    } while (0)
    if (b.tile_sets == 1 && b.tile_waves == 4) ITAK_TILES(1, 4);
    else if (b.tile_sets == 1) ITAK_TILES(1, 8);
    else if (b.tile_waves == 4) ITAK_TILES(2, 4);
    else ITAK_TILES(2, 8);
#undef ITAK_TILES
    return e;
}

}  // namespace itak
