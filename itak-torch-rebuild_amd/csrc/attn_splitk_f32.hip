// f32 pools at head_dim 64 and 128: the planner of the row-major split-K launches and this kernel's
// instantiations for them (attn_splitk_rows_kernel.h).
#include "attn_splitk_rows_kernel.h"

#include <algorithm>

namespace itak {

bool attn_splitk_f32_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows) {
    return g.v_block == 0 && (g.head_dim == 128 || g.head_dim == 64) && group >= 1 && max_rows >= 1;
}
// Blocks up to which every context of a batch stays whole: a merge launch costs 2 to 3 us and more
// the more there is to merge, against the rounds of blocks that eight wavefronts walk (eight blocks
// a round on blocked planes, four on row-major ones; a round costs 0.5 us there and 1 to 2 us here).
// `units` = workgroups when whole; beyond the compute units they queue.
// Blocked, head_dim 64 to 112, us a layer, split -> whole: one slot at 300 / 450 7.8 / 7.9 -> 5.7 / 6.8, 4
// slots at 600 8.8 -> 7.1. f32, head_dim 64, six rows at 200 9.1 -> 7.8, 8 slots of them at 500 15.0 -> 12.3;
// head_dim 128, 12 rows, 8 slots at 500 29.4 -> 20.7 (one slot, one row at 200 10.8 -> 11.2, at 450 17.0).
// Checked with every shape forced whole and forced split, six head layouts (32/4, 32/8, 16/4, 24/8, 8/8 and
// 8/1), 1, 4 and 16 slots at 120 to 1,500 positions: within 5 % of the better on nine of ten, 2 % behind
// on average. Where it is far off, contexts just past the line of launches of many units are split that
// were better whole: f32, head_dim 64, 16 slots of six rows at 600 24.9 against 14.1, f16, head_dim 64, one
// row of each at 900, 8 KV heads, 14.0 against 10.5.
static uint32_t whole_limit(const PoolGeom &g, int elem_f16, uint64_t units, uint32_t vectors, bool may_eight, uint64_t cus) {
    const uint32_t d = g.head_dim;
    if (!may_eight || units > cus) return vectors > 16 ? 0 : g.v_block ? (d <= 128 ? 12 : 8) : elem_f16 || d <= 64 ? 8 : 4;
    if (g.v_block) return units >= 16 ? 24 : 16;
    if (d <= 64) return units >= 96 ? 16 : 8;
    return units >= 128 ? 16 : elem_f16 || units >= 32 ? 8 : 4;
}

// Fills splits / keys_per_split / block0 / ws0 (slot, rows, pos0, q_row0, kv_len, kv_lo are
// set) and returns the number of partials. Every (item, KV head) is cut into equal runs of at
// most T blocks, T the smallest run for which the batch is at most groups_per_cu workgroups per
// compute unit, and never shorter than one block per wavefront.
uint32_t attn_splitk_f32_plan(const PoolGeom &g, int elem_f16, AttnBatch &b, uint32_t q_heads, uint32_t groups_per_cu) {
    const uint64_t cus = compute_units();
    uint64_t capacity = groups_per_cu * cus;
    const uint32_t group = q_heads / g.kv_heads;
    auto units_of = [&](const AttnItem &it) {
        return uint64_t(g.kv_heads) * ((uint64_t(it.rows) * group + 15) / 16);
    };
    auto groups_at = [&](uint64_t run) {
        uint64_t groups = 0;
        for (uint32_t i = 0; i < b.n; ++i)
            groups += units_of(b.item[i]) * std::max<uint64_t>((item_block_count(b.item[i]) + run - 1) / run, 1);
        return groups;
    };
    uint64_t blocks = 0, units = 0;
    uint32_t most = 0, vectors = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        units += units_of(b.item[i]);
        blocks += units_of(b.item[i]) * item_block_count(b.item[i]);
        most = std::max(most, item_block_count(b.item[i]));
        vectors = std::max(vectors, b.item[i].rows * group);
    }
    // Eight wavefronts: whole contexts of more than one round of four, and, on row-major planes, one
    // tile of vectors over up to 16 blocks per compute unit, where half a block per wavefront halves the
    // chain of f32 products (32 cycles each) and one workgroup per compute unit the partials
    // (one row at 12,000, head_dim 64 / 128 11.5 / 18.3 -> 10.1 / 14.6 us a layer; several tiles at
    // 1,000 to 3,000 lose up to a third).
    const bool may_eight = g.head_dim <= 128;
    const bool whole = most <= whole_limit(g, elem_f16, units, vectors, may_eight, cus);
    b.on_eight = may_eight && (whole ? most > (g.v_block ? 4u : 2u)
                                     : !g.v_block && vectors <= 16 && groups_at(4) <= 4 * cus);
    // Row-major launches that two blocks a workgroup spread over no more than the compute units: four
    // wavefronts, half a block each. A block is 4,096 cycles of f32 products at head_dim 128, whoever
    // shares them.
    b.half_blocks = !g.v_block && !whole && most <= 128 && groups_at(2) <= cus;
    if (b.half_blocks) b.on_eight = 0;
    if (b.on_eight || b.half_blocks) capacity = cus;
    uint64_t T = std::max<uint64_t>((blocks + capacity - 1) / capacity, b.half_blocks ? 2 : 4);
    if (whole) T = std::max<uint64_t>(T, most);
    // (Units that alone outnumber the device are left whole: nothing is gained by splitting.)
    while (T < most && T < 4096 && groups_at(T) > capacity) ++T;
    uint32_t block0 = 0, ws0 = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        AttnItem &it = b.item[i];
        const uint32_t nblocks = item_block_count(it);
        it.splits = std::max<uint32_t>(uint32_t((nblocks + T - 1) / T), 1);
        const uint32_t bps = std::max<uint32_t>((nblocks + it.splits - 1) / it.splits, 1);
        it.splits = std::max<uint32_t>((nblocks + bps - 1) / bps, 1);
        it.keys_per_split = bps * kBlockKeys;
        it.splits_magic = 0;
        it.block0 = block0;
        it.ws0 = ws0;
        block0 += uint32_t(units_of(it)) * it.splits;
        if (it.splits > 1) ws0 += it.rows * q_heads * it.splits;
    }
    b.total_blocks = block0;
    b.rows_per_block = 0;
    return ws0;
}

hipError_t launch_attn_splitk_f32(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  hipStream_t stream) {
    if (b.total_blocks == 0) return hipSuccess;
    // One tile of vectors per KV head in every item: each K/V row is read by one workgroup.
    // (And only where the keys and values would not stay in the last-level cache anyway: a pool
    // small enough to live there reads faster without the hint, 33.9 against 37.2 us for 4 slots
    // of 8192 rows on two layers.)
    bool single = p.kv_streams != 0;
    for (uint32_t i = 0; i < b.n; ++i) single = single && b.item[i].rows * p.group <= 16;
#define ITAK_LAUNCH_F32_W(D, STREAM, W, HALF)                                                             \
    ITAK_DISPATCH_BATCH(b.n, (launch_kernel(attn_splitk_rows_kernel<float, D, true, 1, STREAM, W, HALF, N>, b.total_blocks, \
                                            W * 64, 0, stream, p, AttnBatchT<N>(b), total_partials)))
#define ITAK_LAUNCH_F32(D, STREAM)                          \
    do {                                                    \
        if (b.on_eight)                                     \
            ITAK_LAUNCH_F32_W(D, STREAM, 8, true);          \
        else if (b.half_blocks)                             \
            ITAK_LAUNCH_F32_W(D, STREAM, 4, true);          \
        else                                                \
            ITAK_LAUNCH_F32_W(D, STREAM, 4, false);         \
    } while (0)
    if (p.g.head_dim == 64) {
        if (single) ITAK_LAUNCH_F32(64, true);
        else ITAK_LAUNCH_F32(64, false);
    } else {
        if (single) ITAK_LAUNCH_F32(128, true);
        else ITAK_LAUNCH_F32(128, false);
    }
#undef ITAK_LAUNCH_F32
#undef ITAK_LAUNCH_F32_W
    return hipGetLastError();
}

}  // namespace itak
