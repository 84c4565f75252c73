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
// were better whole: f16, head_dim 64, one row of each slot at 900, 8 KV heads, 14.0 against 10.5; blocks of
// several tiles (f32, head_dim 64, 16 slots of six rows at 600, 24.9 against 14.1) go by cut_costs below.
static uint32_t whole_limit(const PoolGeom &g, int elem_f16, uint64_t units, uint32_t vectors, bool may_eight, uint64_t cus) {
    const uint32_t d = g.head_dim;
    if (!may_eight || units > cus) return vectors > 16 ? 0 : g.v_block ? (d <= 128 ? 12 : 8) : elem_f16 || d <= 64 ? 8 : 4;
    if (g.v_block) return units >= 16 ? 24 : 16;
    if (d <= 64) return units >= 96 ? 16 : 8;
    return units >= 128 ? 16 : elem_f16 || units >= 32 ? 8 : 4;
}

// What a launch of several tiles a KV head takes, in microseconds a layer, by how it is cut and walked:
// the launch, every workgroup a compute unit runs in turn, a wavefront's rounds of them, the chain of
// the longest, all blocks over the compute units, and the merge with its partials.
struct CutCost {
    float launch, group, round, chain, block, merge, partial;
    float of(uint64_t workgroups, uint64_t rounds, uint64_t blocks, uint64_t partials, uint32_t d, uint64_t cus) const {
        const float turns = float((workgroups + cus - 1) / cus), wide = float(d) / 128;
        return launch + turns * wide * (group + round * float(rounds)) + chain * float(rounds) +
               block * float(blocks) / float(cus) + (partials ? merge + partial * 1e-6f * float(partials) * float(d) : 0);
    }
};
// Four wavefronts, eight, and four that take half a block each; a launch of 0 = not a form of the kernel.
struct CutCosts {
    CutCost four, eight, half;
};
// Fitted over 8,200 launches of more than 16 vectors a KV head, each timed over counts and forms with the
// keys and values out of the caches (six head layouts, 1 to 8 slots, 2 to 200 rows, 30 to 16,000 keys). The
// plan by whole_limit's line and the device's fill was 19 % behind the best of them on average beyond
// head_dim 128, 4 % on narrower blocked planes, 7 and 5 % on f32 planes of 64 and 128; by these 1, 2, 3 and 3 %.
// The even fill is far off for contexts just past the line, which it splits whatever the merge costs:
// 3 slots of 38 rows at 198, head_dim 192, 32 Q / 4 KV heads 31.6 -> 13.9 us, 4 of 21 at 839 38.2 -> 21.6;
// head_dim 80, 7 slots of 13 rows at 911 24.4 -> 14.6; f32, head_dim 64, 8 of 12 at 845 27.7 -> 17.2.
// Row-major f16 planes keep the line: their estimates missed by up to a half. (`merge`, and the split figures of whole_limit, are
// of a merge launch that asked for eight partials a lane whatever there were; it takes 0.3 to 0.5 us less now.)
static const CutCosts *cut_costs(const PoolGeom &g, int elem_f16) {
    static const CutCosts kBlocked{{5.04f, 2.56f, 0.55f, 0.49f, 0.137f, 3.17f, 2.85f},
                                   {4.98f, 4.00f, 1.04f, 0.34f, 0.169f, 3.07f, 5.64f},
                                   {}};
    static const CutCosts kBlockedWide{{5.74f, 2.67f, 0.90f, 0.04f, 0.256f, 3.15f, 1.95f}, {}, {}};
    static const CutCosts kF32x64{{3.48f, 0.50f, 0.97f, 1.53f, 0.205f, 3.12f, 4.61f},
                                  {3.86f, 0.43f, 1.96f, 0.46f, 0.167f, 3.09f, 5.78f},
                                  {3.64f, 0.00f, 0.71f, 0.67f, 0.177f, 3.15f, 5.13f}};
    static const CutCosts kF32x128{{4.20f, 1.02f, 1.62f, 1.25f, 0.326f, 2.70f, 1.92f},
                                   {2.67f, 2.87f, 1.64f, 0.67f, 0.423f, 3.09f, 1.51f},
                                   {4.27f, 0.79f, 0.96f, 0.51f, 0.299f, 2.76f, 2.07f}};
    if (elem_f16) return !g.v_block ? nullptr : g.head_dim <= 128 ? &kBlocked : &kBlockedWide;
    return g.head_dim == 64 ? &kF32x64 : g.head_dim == 128 ? &kF32x128 : nullptr;
}

// Fills splits / keys_per_split / block0 / ws0 (slot, rows, pos0, q_row0, kv_len, kv_lo are
// set) and returns the number of partials. Every (item, KV head) is cut into equal runs of at
// most T blocks, T the smallest run for which the batch is at most groups_per_cu workgroups per
// compute unit, and never shorter than one block per wavefront; blocks of
// several tiles by what the cuts are estimated to take (cut_costs). `partial_bytes` = the most the partials of
// such a cut may take (0 = any). `may_part` = false keeps one-row steps from attn_parts_halves.hip.
uint32_t attn_splitk_f32_plan(const PoolGeom &g, int elem_f16, AttnBatch &b, uint32_t q_heads, uint32_t groups_per_cu,
                              uint64_t partial_bytes, bool may_part) {
    uint32_t in_parts = 0;
    if (elem_f16 && may_part && attn_parts_halves_plan(g, b, q_heads, &in_parts)) return in_parts;
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
    uint64_t blocks = 0, units = 0, rows = 0;
    uint32_t most = 0, vectors = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        units += units_of(b.item[i]);
        blocks += units_of(b.item[i]) * item_block_count(b.item[i]);
        most = std::max(most, item_block_count(b.item[i]));
        vectors = std::max(vectors, b.item[i].rows * group);
        rows += b.item[i].rows;
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
    // Several tiles over contexts of about one length, on up to four workgroups a compute unit: another cut is
    // taken where it is estimated to be 8 % ahead (by less, one launch in 20 lost more than it gained).
    const CutCosts *costs = vectors > 16 && units <= 4 * cus && 4 * blocks >= 3 * units * most ? cut_costs(g, elem_f16) : nullptr;
    if (costs && most > 0) {
        const uint64_t partial = uint64_t(g.head_dim + 2) * sizeof(float);
        auto cost_of = [&](const CutCost &c, uint64_t run, uint32_t per_round) {
            const uint64_t count = (most + run - 1) / run;
            return c.of(units * count, (run + per_round - 1) / per_round, blocks, count > 1 ? rows * q_heads * count : 0,
                        g.head_dim, cus);
        };
        auto per_round = [&](bool eight, bool half) { return half ? 2u : eight && g.v_block ? 8u : 4u; };
        const uint64_t now = std::min<uint64_t>(T, most);
        uint64_t parts = 0;
        for (uint32_t i = 0; i < b.n; ++i) {
            const uint64_t count = (item_block_count(b.item[i]) + now - 1) / now;
            if (count > 1) parts += b.item[i].rows * q_heads * count;
        }
        // (A step whose partials outgrow the caller's workspace is left as it is.)
        const bool fits = !partial_bytes || parts * partial <= partial_bytes;
        float best = cost_of(b.half_blocks ? costs->half : b.on_eight ? costs->eight : costs->four, now,
                             per_round(b.on_eight, b.half_blocks)) / 1.08f;
        for (uint32_t count = 1; fits && count <= 64 && (count == 1 || units * count <= 4 * cus); count += 1 + count / 4) {
            const uint64_t run = (most + count - 1) / count;
            if (count > 1 && (run < 2 || (partial_bytes && rows * q_heads * count * partial > partial_bytes))) break;
            for (uint32_t form = 0; form < 3; ++form) {
                const CutCost &c = form == 0 ? costs->four : form == 1 ? costs->eight : costs->half;
                if (c.launch == 0) continue;
                const float cost = cost_of(c, run, per_round(form == 1, form == 2));
                if (cost >= best) continue;
                best = cost;
                T = run;
                b.on_eight = form == 1;
                b.half_blocks = form == 2;
            }
        }
    }
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
