// f32 pools at head_dim 64 and 128: the planner of the row-major split-K launches and this kernel's
// instantiations for them (attn_splitk_rows_kernel.h).
#include "attn_splitk_rows_kernel.h"

#include <algorithm>

namespace itak {

bool attn_splitk_f32_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows) {
    return g.v_block == 0 && (g.head_dim == 128 || g.head_dim == 64) && group >= 1 && max_rows >= 1;
}
// Steps of up to 16 query vectors per KV head bring their rows along: every workgroup that
// reaches the new positions copies all of them in, which is nothing for a row or two and would
// be the whole chunk for a prefill.
bool attn_splitk_f32_appends(const PoolGeom &g, uint32_t group, uint32_t max_rows) {
    return attn_splitk_f32_supports(g, group, max_rows) && max_rows * group <= 16;
}

// Fills splits / keys_per_split / block0 / ws0 (slot, rows, pos0, q_row0, kv_len, kv_lo are
// set) and returns the number of partials. Every (item, KV head) is cut into equal runs of at
// most T blocks, T the smallest run for which the batch is at most groups_per_cu workgroups per
// compute unit, and never shorter than one block per wavefront.
uint32_t attn_splitk_f32_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, uint32_t groups_per_cu, uint32_t whole_blocks) {
    const uint64_t capacity = uint64_t(groups_per_cu) * compute_units();
    const uint32_t group = q_heads / g.kv_heads;
    auto units_of = [&](const AttnItem &it) {
        return uint64_t(g.kv_heads) * ((uint64_t(it.rows) * group + 15) / 16);
    };
    uint64_t blocks = 0;
    for (uint32_t i = 0; i < b.n; ++i) blocks += units_of(b.item[i]) * item_block_count(b.item[i]);
    uint64_t T = std::max<uint64_t>((blocks + capacity - 1) / capacity, uint64_t(kWavesRows));
    // A short step's short contexts stay whole (one tile of vectors per KV head): a merge launch costs
    // 2 to 3 us, a wavefront's second 32-key block 1 us on the f32 pipe at head_dim 64, twice that at
    // 128, half of it on the f16 pipe. One row at 200 positions, 1 slot: f32 at head_dim 64 8.1 -> 7.5
    // us a layer (at 128 10.1 -> 10.2), f16 at 80 8.6 -> 6.5 and, at 300 positions, 8.4 -> 7.5.
    uint32_t most = 0, most_vectors = 0;
    for (uint32_t i = 0; i < b.n; ++i) {
        most = std::max(most, item_block_count(b.item[i]));
        most_vectors = std::max(most_vectors, b.item[i].rows * group);
    }
    if (most_vectors <= 16 && most <= whole_blocks) T = std::max<uint64_t>(T, most);
    for (;; ++T) {
        uint64_t groups = 0;
        for (uint32_t i = 0; i < b.n; ++i) {
            const uint64_t nb = item_block_count(b.item[i]);
            groups += units_of(b.item[i]) * std::max<uint64_t>((nb + T - 1) / T, 1);
        }
        // (Units that alone outnumber the device are left whole: nothing is gained by splitting.)
        if (groups <= capacity || T >= blocks || T >= 4096) break;
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
#define ITAK_LAUNCH_F32(D, STREAM)                                                                        \
    ITAK_DISPATCH_BATCH(b.n, (launch_kernel(attn_splitk_rows_kernel<float, D, true, 2, STREAM, N>, b.total_blocks, \
                                            kWavesRows * 64, 0, stream, p, AttnBatchT<N>(b), total_partials)))
    if (p.g.head_dim == 64) {
        if (single) ITAK_LAUNCH_F32(64, true);
        else ITAK_LAUNCH_F32(64, false);
    } else {
        if (single) ITAK_LAUNCH_F32(128, true);
        else ITAK_LAUNCH_F32(128, false);
    }
#undef ITAK_LAUNCH_F32
    return hipGetLastError();
}

}  // namespace itak
