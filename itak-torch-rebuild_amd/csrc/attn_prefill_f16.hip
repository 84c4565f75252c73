// The block kernel's host side: which launches it takes, their plan, and the head_dim 128
// instantiations (attn_prefill_f16_kernel.h has the kernel).
#include "attn_prefill_f16_kernel.h"

#include <cmath>

// Timeline marks of attn_prefill_f16_kernel: 0 first instruction, 1 addresses known, 2 first
// blocks and Q requested, 3 Q converted (it has arrived), 4 first block multiplied, 5 last block
// multiplied, 6 output or partials issued, 11 all done; of the first block: 7 its loads have
// landed, 8 past the barrier, 9 new rows written over it.
ITAK_TIMELINE_READER(itak_timeline_read_prefill)

namespace itak {

// A launch may bring its items' new rows along (AttnParams::k_new / v_new) when it takes the
// one-tile form and no item has more than kFuseRows rows.
bool attn_prefill_f16_appends(const PoolGeom &g, uint32_t group, uint32_t most_rows,
                              uint32_t most_blocks) {
    return attn_prefill_f16_supports(g, group) && most_rows <= uint32_t(fuse_rows(int(g.head_dim))) &&
           most_rows * padded_group(group) <= 512 && most_blocks <= kFuseBlocks;
}

bool attn_prefill_f16_supports(const PoolGeom &g, uint32_t group) {
    return g.v_block == kVBlock &&
           (g.head_dim == 64 || g.head_dim == 96 || g.head_dim == 128 || g.head_dim == 256) &&
           group >= 1 && group <= 16;
}

// Key blocks one (row tile, KV head) unit of an item walks at most: everything up to the
// item's end on a global layer, the window of its first row plus its own rows on a windowed
// one (the kernel starts each workgroup at its own first visible block).
static uint32_t unit_block_count(const AttnItem &it, uint32_t rows_per_group, uint32_t window) {
    const uint32_t all = item_block_count(it);
    if (window == 0) return all;
    const uint32_t span = window + std::min(rows_per_group, it.rows) + 2 * kBlockKeys - 2;
    return std::min(all, span / kBlockKeys);
}

// What a plan costs in microseconds, as a sum of what its parts measured; the planner takes the
// cheapest. A wavefront holds one or two 16-vector tiles (`tiles`), so a workgroup 64 or 128 vectors,
// and every (row tile, KV head) unit's context is cut into equal runs.
//
// The walk. Alone on its compute unit a workgroup takes `alone` a block: with three blocks in flight
// one tile waits for memory, two for the chain of their products. Two to a compute unit share it,
// `shared` a block of each: less than twice as much, since the waiting overlaps (at head_dim 256 there is
// room for one, and the second comes after it). More workgroups than the device holds at once queue
// behind one another, the longest first. Splits cost a second launch (`merge`) and their partials, written
// and read again at `rate`.
//
// Head_dim 128: fitted on 9 to 1,200 rows over contexts of 0 to 30,000 at 1, 4 and 8 KV heads, global and
// windowed, with every count of tiles and splits timed for each: the pick is 1.4 % behind the best of
// them on average; the rules by size it replaces, which also had an eight-stage ring for launches of one
// workgroup per compute unit (never the best of a shape), were 7 % behind. The other head dims have
// figures of their own, fitted the same way on 4 to 200 rows, 1 to 16 slots and contexts of 90 to 9,000, with
// what the launch reads as a second bound: a block does not take half the time at half the head_dim, and a
// merge launch is another kernel there, with less of a rate. With the figures of 128 scaled by the head_dim,
// windows and contexts of a few hundred positions stayed whole and runs at 256 were never shorter than eight
// blocks: 5 to 14 % behind the best plan, up to 65; with their own 1.2 to 2 %, up to 23. Us a layer: head_dim
// 256, four rows at 400 20.3 -> 12.5; head_dim 96, four rows on a window of 512 14.0 -> 10.1; head_dim 64, 5
// slots of seven rows at 1,100 17.1 -> 14.0. (The other way: head_dim 64, 16 slots of seven at 1,100 17.8 ->
// 20.9.) `merge` is of a merge launch that asked for eight partials a lane whatever there were; it takes 0.3 to 0.8 us
// less now.
struct PlanCost {
    float alone[2], shared[2], merge;
    float rate;              // bytes a microsecond
    float hidden, read_rate; // what a launch reads once, beside that part of its walk (0 = not priced)
};
static const PlanCost &plan_cost(uint32_t head_dim) {
    static constexpr PlanCost k64 = {{0.30f, 0.43f}, {0.47f, 0.78f}, 4.1f, 1.25e6f, 0.14f, 16.2e6f};
    static constexpr PlanCost k96 = {{0.41f, 0.56f}, {0.58f, 0.67f}, 4.2f, 1.14e6f, 0.16f, 8.0e6f};
    static constexpr PlanCost k128 = {{0.345f, 0.56f}, {0.6f, 0.83f}, 4.5f, 2.5e6f, 0.0f, 0.0f};
    static constexpr PlanCost k256 = {{0.70f, 1.20f}, {2.79f, 4.74f}, 4.7f, 5.8e6f, 0.38f, 5.2e6f};
    return head_dim <= 64 ? k64 : head_dim <= 96 ? k96 : head_dim <= 128 ? k128 : k256;
}

struct Shape {
    uint64_t groups = 0;         // workgroups
    uint64_t blocks = 0;         // blocks all of them walk
    float longest = 0.0f;        // and one of them at most
    uint64_t partial_bytes = 0;
    uint64_t read_bytes = 0;     // keys and values, once
};
// An item's blocks per unit and its units, for the tiles at hand.
struct ItemWork {
    uint32_t blocks, units;
};
static Shape shape_of(const PoolGeom &g, const AttnBatch &b, const ItemWork *work, uint32_t q_heads, uint32_t window,
                      uint32_t T, bool appends) {
    Shape s;
    for (uint32_t i = 0; i < b.n; ++i) {
        const uint32_t rows = b.item[i].rows, nb = work[i].blocks, units = work[i].units;
        const uint32_t splits = std::max((nb + T - 1) / T, 1u);
        s.groups += uint64_t(units) * splits;
        // (A causal row tile ends where its rows do.)
        s.blocks += uint64_t(units) * (nb - (window ? 0 : std::min(rows / 64, nb / 2)));
        // (The workgroups that convert and place new rows walk that much less, see below.)
        const float run = float(nb + (appends ? rows / 8 + 1 : 0)) / float(splits);
        s.longest = std::max(s.longest, g.head_dim == 128 ? run : std::ceil(run));  // (as each was fitted)
        s.read_bytes += uint64_t(g.kv_heads) * nb * stage_bytes(int(g.head_dim));
        if (splits > 1) s.partial_bytes += uint64_t(rows) * q_heads * splits * (g.head_dim + 2) * 4;
    }
    return s;
}
static float cost_of(const PlanCost &cost, const Shape &s, int tiles, uint64_t per_cu) {
    const float alone = cost.alone[tiles - 1], shared = cost.shared[tiles - 1];
    float walk = s.longest * alone;
    if (s.groups > 2 * per_cu)
        walk = std::max(walk, 0.5f * walk + float(s.blocks) / float(2 * per_cu) * shared);
    else if (s.groups > per_cu)
        walk = std::max(walk, 0.27f * walk + 0.73f * float(s.blocks) / float(s.groups) * shared);
    if (cost.read_rate > 0.0f) walk = std::max(walk, cost.hidden * walk + float(s.read_bytes) / cost.read_rate);
    return walk + (s.partial_bytes ? cost.merge + float(s.partial_bytes) / cost.rate : 0.0f);
}

// Fills splits / keys_per_split / block0 / ws0 and the tiles for a batch (slot, rows, pos0, q_row0,
// kv_len already set) and returns the number of partials the launch will write.
uint32_t attn_prefill_f16_plan(const PoolGeom &g, AttnBatch &b, uint32_t group, uint32_t q_heads,
                               uint32_t window, bool appends) {
    const uint64_t per_cu = compute_units();
    const uint32_t gp = padded_group(group);
    uint32_t nvec = 0, T = 1;
    for (uint32_t i = 0; i < b.n; ++i) nvec = std::max(nvec, b.item[i].rows * gp);
    float least = INFINITY;
    // Launches that bring their rows along have one tile; so have those of up to 64 vectors, which a
    // second would leave empty. The queries as two halves have registers in the two-tile form only.
    const int first = b.two_halves ? 2 : 1, last = !b.two_halves && (appends || nvec <= 64) ? 1 : 2;
    // Splits of the longest item that are tried; every second count on large batches (a try costs the
    // host 10 ns an item).
    constexpr uint8_t kCounts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 56, 64};
    for (int tiles = first; tiles <= last; ++tiles) {
        const uint32_t rows_per_group = uint32_t(tiles * kWaves * 16) / gp;
        ItemWork work[kMaxBatchItems];
        uint32_t most = 0, before = 0;
        for (uint32_t i = 0; i < b.n; ++i) {
            work[i] = {unit_block_count(b.item[i], rows_per_group, window),
                       g.kv_heads * ((b.item[i].rows + rows_per_group - 1) / rows_per_group)};
            most = std::max(most, work[i].blocks);
        }
        for (uint32_t c = 0; c < sizeof(kCounts); c += b.n > 8 && c ? 2 : 1) {
            const uint32_t run = std::max((most + kCounts[c] - 1) / kCounts[c], 1u);
            if (run == before) continue;
            // (A run asks for three blocks more than it walks, at head_dim 256 of 32 KiB each. One-row steps there
            // are many short units and mind: 4 slots over 1,500, 8 KV heads, in runs of six 22.8 us, of eight 17.8.
            // Steps of several rows do not: one slot of four rows at 400, 4 KV heads, 20.4 -> 12.5 with runs of two.)
            if (c && run < (g.head_dim > 128 && nvec <= 16 ? 8u : 2u)) break;
            before = run;
            const Shape shape = shape_of(g, b, work, q_heads, window, run, appends);
            if (b.partial_limit && shape.partial_bytes > b.partial_limit) break;  // (the whole contexts come first and have none)
            const float cost = cost_of(plan_cost(g.head_dim), shape, tiles, per_cu);
            if (cost < least) {
                least = cost;
                T = run;
                b.tiles = tiles;
            }
        }
    }
    const uint32_t rows_per_group = b.tiles * kWaves * 16 / gp;
    b.plan_cost = least;
    b.fold_units = 0;
    uint32_t block0 = 0, ws0 = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        AttnItem &it = b.item[i];
        const uint32_t nblocks = unit_block_count(it, rows_per_group, window);
        const uint32_t units = g.kv_heads * ((it.rows + rows_per_group - 1) / rows_per_group);
        uint32_t splits = std::max<uint32_t>(uint32_t((nblocks + T - 1) / T), 1);
        uint32_t bps = std::max<uint32_t>((nblocks + splits - 1) / splits, 1);
        // A launch that appends its own rows: the workgroups of a unit's last split convert
        // the new rows and write them over their last blocks, about a block's time for every
        // eight rows, and the launch ends with them; their run is made that much shorter and
        // the other splits share the difference.
        if (appends && splits > 1) {
            const uint32_t extra = std::min<uint32_t>(it.rows / 8 + 1, bps / 2);
            const uint32_t longer = (nblocks + extra + splits - 1) / splits;
            if (uint64_t(splits - 1) * longer < nblocks) bps = longer;
        }
        splits = std::max<uint32_t>((nblocks + bps - 1) / bps, 1);
        it.splits = splits;
        it.keys_per_split = bps * kBlockKeys;
        it.splits_magic = 0;
        it.block0 = block0;
        it.ws0 = ws0;
        block0 += units * splits;
        if (splits > 1) ws0 += it.rows * q_heads * splits;
    }
    b.total_blocks = block0;
    b.rows_per_block = rows_per_group;
    // One unsplit item whose row tiles see different numbers of blocks (no window) and whose
    // workgroups are all resident from the start, two to a compute unit: fold the second run
    // (see the kernel; 2048 rows without a prefix 64.9 -> 61.6 us per layer). With more runs
    // the later workgroups go wherever one ends, which balances better unfolded (4096 and 8192
    // rows measured 1 to 3 % slower folded).
    if (b.n == 1 && b.item[0].splits == 1 && window == 0 && block0 > per_cu &&
        block0 <= 2 * per_cu && per_cu % g.kv_heads == 0)
        b.fold_units = uint32_t(per_cu);
    return ws0;
}

hipError_t launch_attn_prefill_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                   hipStream_t stream) {
    if (b.total_blocks == 0) return hipSuccess;
    const bool one = b.tiles == 1;
    if (p.k_new && !one) return hipErrorInvalidValue;  // only the one-tile form appends
    if (b.two_halves) return launch_attn_prefill_f16_qlo(p, b, total_partials, stream);
    if (p.g.head_dim == 128) return launch_prefill_head_dim<128, true>(p, b, total_partials, one, stream);
    return launch_attn_prefill_f16_dims(p, b, total_partials, one, stream);
}

}  // namespace itak
