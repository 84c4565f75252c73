// Shared declarations between the host logic (pool.hip) and the kernel files.
// Nothing here is part of the public ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace itak {

// A kernel launch without the triple-chevron form's detour (the configuration pushed to and popped
// from the runtime's per-thread stack): 1.95 us of host time instead of 2.45. Errors are the
// runtime's last error, as after that form.
template <typename... P>
inline void launch_kernel_args(void (*kernel)(P...), dim3 grid, dim3 block, uint32_t lds, hipStream_t stream,
                               const P &...args) {
    void *at[] = {const_cast<void *>(static_cast<const void *>(&args))...};
    (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, stream);
}
template <typename... P, typename... A>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, uint32_t lds, hipStream_t stream, const A &...args) {
    static_assert(sizeof...(P) == sizeof...(A), "one argument per parameter");
    launch_kernel_args<P...>(kernel, grid, block, lds, stream, static_cast<const P &>(args)...);
}
// A kernel without parameters.
inline void launch_kernel(void (*kernel)(), dim3 grid, dim3 block, uint32_t lds, hipStream_t stream) {
    (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, nullptr, lds, stream);
}

// Compute units of the current device, asked of the runtime once per device.
uint32_t compute_units();

// Device layout of the KV pool, in elements of the storage type. One "plane" is the
// rows of one (layer, slot, side, kv_head): capacity x head_dim elements, contiguous,
// so a workgroup that streams one KV head reads one unbroken run of memory.
//   plane(layer, slot, side, head) =
//     layer*layer_stride + slot*slot_stride + side*side_stride + head*head_stride
// side 0 = keys, 1 = values. With v_block == 0 both are row-major (row*head_dim + d).
// With v_block == 32 (f16 pools whose head_dim is a multiple of 16) both are stored in
// blocks of 32 rows laid out as the MFMA kernels consume them, so that every operand load
// of a wavefront is 64 lanes x 16 bytes of contiguous memory:
//   values: block transposed, element (row, d) at
//       (row/32)*32*head_dim + d*32 + row%32
//     (a lane's 8 consecutive rows of one channel are 16 contiguous bytes);
//   keys: 16-byte pieces of 8 channels, grouped by MFMA tile t and channel chunk c, element
//     (row, d) with kk = row%32, t = (kk/4)%2, i = (kk/8)*4 + kk%4, c = d/8 at
//       (row/32)*32*head_dim + ((t*(head_dim/8) + c)*16 + i)*8 + d%8
//     (tile t holds the 16 rows whose scores one lane group receives as 8 consecutive
//     keys; the lanes (chunk c, row i) of one load instruction are adjacent in memory).
struct PoolGeom {
    uint32_t kv_heads;
    uint32_t head_dim;
    uint32_t capacity;  // rows per plane (a multiple of 32 when v_block != 0)
    uint32_t max_slots;
    uint32_t v_block;   // 0 or 32
    uint32_t pad;
    uint64_t head_stride;   // capacity * head_dim
    uint64_t side_stride;   // kv_heads * head_stride
    uint64_t slot_stride;   // 2 * side_stride
    uint64_t layer_stride;  // max_slots * slot_stride
};

constexpr uint32_t kVBlock = 32;

// Element offset of (row, d) inside a value plane.
__host__ __device__ inline uint64_t v_offset(const PoolGeom &g, uint32_t row, uint32_t d) {
    if (g.v_block == 0) return uint64_t(row) * g.head_dim + d;
    return uint64_t(row / kVBlock) * (kVBlock * g.head_dim) + uint64_t(d) * kVBlock + row % kVBlock;
}

// Element offset of (row, d) inside a key plane.
__host__ __device__ inline uint64_t k_offset(const PoolGeom &g, uint32_t row, uint32_t d) {
    if (g.v_block == 0) return uint64_t(row) * g.head_dim + d;
    const uint32_t kk = row % kVBlock;
    const uint32_t t = (kk >> 2) & 1, i = (kk >> 3) * 4 + (kk & 3);
    return uint64_t(row / kVBlock) * (kVBlock * g.head_dim) +
           ((t * (g.head_dim / 8) + d / 8) * 16 + i) * 8 + d % 8;
}

// Element offset inside a plane of either side.
__host__ __device__ inline uint64_t kv_offset(const PoolGeom &g, uint32_t side, uint32_t row,
                                              uint32_t d) {
    return side ? v_offset(g, row, d) : k_offset(g, row, d);
}

// f32 -> f16 bits, round-to-nearest-even, overflow to infinity, subnormals rounded, and
// every NaN stored as sign|0x7e00: the rule of f32_to_f16_bits in
// crates/wgpu-compute/src/kernels/k1_q4k_gemv.rs:285-329. v_cvt_f16_f32 implements all of
// it except the NaN payload, which is replaced explicitly.
__device__ __forceinline__ uint16_t f32_to_f16_bits(float x) {
    _Float16 h = static_cast<_Float16>(x);
    uint16_t bits = __builtin_bit_cast(uint16_t, h);
    uint32_t in = __builtin_bit_cast(uint32_t, x);
    if ((in & 0x7fffffffu) > 0x7f800000u) {
        bits = static_cast<uint16_t>(((in >> 16) & 0x8000u) | 0x7e00u);
    }
    return bits;
}

constexpr int kMaxBatchItems = 64;

// ---- append ---------------------------------------------------------------------
struct AppendItem {
    uint32_t slot;
    uint32_t rows;
    uint32_t pos0;      // position of the item's first new row
    uint32_t src_row0;  // row offset of the item inside k_src / v_src
};
struct AppendBatch {
    uint32_t n;
    uint32_t total_rows;
    uint32_t ring;      // storage rows of a windowed layer's ring (position p lives in row p % ring); 0 = row p
    uint32_t pad;
    AppendItem item[kMaxBatchItems];
};
hipError_t launch_append(void *layer_base, int elem_f16, const PoolGeom &g, const AppendBatch &b,
                         const float *k_src, const float *v_src, hipStream_t stream);
// One item's run of rows into blocked f16 planes; sources aligned to 16 bytes, ring (a multiple of
// 32, 0 = none) at least `rows` long.
hipError_t launch_append_chunk(void *layer_base, const PoolGeom &g, uint32_t slot, uint32_t pos0, uint32_t rows,
                               uint32_t ring, const float *k_src, const float *v_src, hipStream_t stream);

// ---- zero fill of dropped rows (truncate scrub, slot reset) ------------------------
struct ZeroItem {
    uint32_t slot;
    uint32_t row_from;
    uint32_t row_to;  // exclusive
    uint32_t pad;
};
struct ZeroBatch {
    uint32_t n;
    uint32_t max_rows;
    ZeroItem item[kMaxBatchItems];
};
hipError_t launch_zero_rows(void *pool_base, int elem_f16, const PoolGeom &g, uint32_t layer_from,
                            uint32_t layer_to, const ZeroBatch &b, hipStream_t stream);

// ---- snapshot restore (gather from [row][kv_head][d] sources into the planes) --------
constexpr int kMaxRestoreLayers = 64;
struct RestoreLayer {
    const void *keys;
    const void *values;
    uint32_t layer;
    uint32_t rows;
    uint32_t first_row;  // destination storage row of source row 0
    uint32_t pad;
};
struct RestoreBatch {
    uint32_t n;
    uint32_t max_rows;
    uint32_t slot;
    uint32_t pad;
    RestoreLayer layer[kMaxRestoreLayers];
};
hipError_t launch_restore(void *pool_base, int dst_f16, int src_f16, const PoolGeom &g,
                          const RestoreBatch &b, hipStream_t stream);

// ---- row readback: planes -> [row][kv_head][d] ---------------------------------------
// Row r of the output is position first_row + r, read from storage row (first_row + r) % ring
// when ring != 0.
hipError_t launch_read_rows(const void *layer_base, int elem_f16, const PoolGeom &g, uint32_t slot,
                            uint32_t first_row, uint32_t rows, uint32_t ring, void *keys_out,
                            void *values_out, hipStream_t stream);

// The same for a stretch of a snapshot's payload: runs of elements of one layer's and side's rows
// ([row][kv_head][d], row 0 at position first_row) to out + out0, as f32 or (out_f16) as they are.
constexpr int kMaxReadRuns = 64;
struct ReadRun {
    uint32_t layer;      // index within its group of planes
    uint32_t side;
    uint32_t first_row;
    uint32_t ring;       // windowed layers: storage rows of the ring; 0 = a global layer
    uint64_t elem0;
    uint64_t count;
    uint64_t out0;
};
struct ReadRuns {
    uint32_t n;
    uint32_t slot;
    ReadRun run[kMaxReadRuns];
};
hipError_t launch_read_runs(const void *base, const void *base_w, int elem_f16, int out_f16, const PoolGeom &g,
                            const PoolGeom &gw, const ReadRuns &b, void *out, hipStream_t stream);

// ---- FNV-1a 64 on the device (fnv_kernels.hip) ------------------------------------------
// *state (device memory) = the hash after `bytes` bytes at `data` (device memory, 16-byte aligned)
// from *state. `bytes` is a multiple of kFnvRun; scratch holds fnv_scratch_bytes(bytes).
constexpr uint32_t kFnvRun = 64;
uint64_t fnv_scratch_bytes(uint64_t bytes);
hipError_t launch_fnv(const void *data, uint64_t bytes, void *scratch, unsigned long long *state, hipStream_t stream);
// The sums of a file's 1 MiB blocks, states[k] = FNV-1a of block k, piece by piece and in order: `bytes` bytes of the
// file from file_at on (a multiple of kFnvRun but for the last piece). A block that begins in the piece starts there; one
// that does not goes on from states[k], which for the file's first block the caller sets.
hipError_t launch_fnv_blocks(const void *data, uint64_t bytes, uint64_t file_at, void *scratch, unsigned long long *states,
                             hipStream_t stream);

// ---- ring rows aside and back (checkpoints deeper than a ring's headroom) -----------------
// Copies rows of windowed layers between their rings and a side buffer that holds, per entry,
// [side][saved_rows][kv_head][d] elements at saved_off: row saved_row0 + r of the buffer is
// position pos0 + r, storage row (pos0 + r) % ring.
struct RingRowsLayer {
    uint32_t layer;       // index among the windowed layers
    uint32_t ring;
    uint32_t pos0;
    uint32_t rows;
    uint32_t saved_row0;
    uint32_t saved_rows;
    uint64_t saved_off;   // elements
};
struct RingRowsBatch {
    uint32_t n;
    uint32_t slot;
    uint32_t max_rows;
    uint32_t pad;
    RingRowsLayer layer[kMaxRestoreLayers];
};
// to_ring = false: rings -> buffer; true: buffer -> rings.
hipError_t launch_ring_rows(void *pool_base_w, int elem_f16, const PoolGeom &gw,
                            const RingRowsBatch &b, void *saved, bool to_ring, hipStream_t stream);

hipError_t launch_convert_f16(const float *src, uint16_t *dst, uint64_t count, hipStream_t stream);
// The other way: `count` halves at src (16-byte aligned, like dst) as f32.
hipError_t launch_widen_f16(const uint16_t *src, float *dst, uint64_t count, hipStream_t stream);
// Host-pointer calls: `bytes` (rounded up to 16) from pinned host memory into device memory by
// a kernel, and a word in pinned host memory set to `value` once everything before it on the
// stream has finished.
hipError_t launch_stage_in(const void *pinned, void *dst, uint64_t bytes, hipStream_t stream);
hipError_t launch_signal_done(uint32_t *pinned_word, uint32_t value, hipStream_t stream);
hipError_t launch_probe_copy(const void *src, void *dst, uint64_t bytes, hipStream_t stream);
hipError_t launch_probe_read(const void *src, uint64_t bytes, hipStream_t stream);
hipError_t launch_probe_empty(hipStream_t stream);
// `iters` trips of 32 f16 MFMAs per wavefront, two workgroups of four wavefronts per compute unit
// (*workgroups receives how many were launched); clocks: two device words or null.
hipError_t launch_probe_mfma(bool random_operands, uint32_t iters, unsigned long long *clocks,
                             uint32_t *workgroups, hipStream_t stream);

// ---- attention preparation (per-head RMSNorm + RoPE of Q and K) and the output gate ------
struct PrepArgs {
    const float *q_in;      // [total_rows][q_heads*head_dim]
    const float *k_in;      // [total_rows][kv_heads*head_dim]
    float *q_out;
    float *k_out;
    const float *q_weight;  // [head_dim] or null: no norm
    const float *k_weight;
    float eps;
    float rope_base;        // > 1 rotates, otherwise no rotation
    // Pair i turns at position * rope_freq[i] radians: rope_base^(-2i/rotary_dim) as the host's
    // libm gives it, which is what the reference's own host computes. Null: the kernel takes
    // the power itself (the device library's may differ in the last bit, and a last bit times
    // the position is what reaches the stored row).
    const double *rope_freq;
    uint32_t interleaved;   // 1: pairs (2i, 2i+1); 0: pairs (i, i + rotary_dim/2)
    uint32_t rotary_dim;
    uint32_t head_dim;
    uint32_t q_heads;
    uint32_t kv_heads;
    uint32_t total_rows;
    uint32_t n;                      // items
    uint32_t row0[kMaxBatchItems];   // first row of item i (rows are laid out item after item)
    uint32_t pos0[kMaxBatchItems];   // position of that row
};
hipError_t launch_attn_prep(const PrepArgs &a, hipStream_t stream);
// dst[0 .. n) = v, which travels as the launch's argument.
constexpr uint32_t kFillDoubles = 64;
struct FillDoubles {
    uint32_t n;
    double v[kFillDoubles];
};
hipError_t launch_fill_doubles(double *dst, const FillDoubles &a, hipStream_t stream);
// out[i] *= sigmoid(gate[i]) (CpuCompute::attn_gate, cpu.rs:657-673).
hipError_t launch_attn_gate(float *out, const float *gate, uint64_t count, hipStream_t stream);

// ---- attention ----------------------------------------------------------------------
// One item = one slot's query rows against that slot's rows of one layer. Query row r
// sits at position pos0 + r unless q_pos is given. A query at position p sees the keys at
// positions max(kv_lo, p + 1 - window) .. min(p, kv_len - 1) (window 0 = no lower bound but
// kv_lo); on a windowed layer position kp lives in storage row kp % (32 * ring_blocks), so
// that 32-position blocks stay whole and in order inside the ring. A workgroup owns (item, row block,
// kv head, split of the key range) and writes either the final output (splits == 1) or
// a partial (m, l, acc[head_dim]) per query vector; a second, small launch merges the
// partials of each (row, Q head). Partials live in `ws`: first total_partials*head_dim
// accumulators, then total_partials (m, l) pairs; the partial of (row, head, split) of
// an item is ws0 + (row*q_heads + head)*splits + split.
struct AttnItem {
    uint32_t slot;
    uint32_t rows;
    uint32_t pos0;
    uint32_t q_row0;        // first row of the item in q / out
    uint32_t kv_len;        // stored rows visible to the item's last query row (exclusive end)
    uint32_t splits;
    uint32_t keys_per_split;
    uint32_t block0;        // first workgroup index of the item
    uint32_t ws0;           // first partial index of the item
    uint32_t splits_magic;  // ceil(2^32 / splits) for splits > 1: x / splits == mulhi(x, magic), x < 2^16. Of a batch that
                            // attn_parts_halves_plan took, of kv_heads * splits in place of splits
    uint32_t kv_lo;         // oldest position any query of the item may see (0 on global layers)
};
// Key blocks (32 positions) an item's queries can touch: [first, end).
__host__ __device__ inline uint32_t item_first_block(const AttnItem &it) { return it.kv_lo / 32; }
__host__ __device__ inline uint32_t item_block_count(const AttnItem &it) {
    return (it.kv_len + 31) / 32 - it.kv_lo / 32;
}
struct AttnBatch {
    uint32_t n;
    uint32_t total_blocks;
    uint32_t rows_per_block;
    uint32_t tiles;      // host side only: column tiles per wavefront in the block kernel's plan
    uint32_t fold_units; // host side only: the block kernel's plan for AttnParams::fold_units
    uint32_t two_halves; // host side only: the block kernel multiplies each query as two f16 halves
    uint32_t on_eight; // host side only: the rows and halves kernels run on eight wavefronts
    uint32_t half_blocks; // host side only: the rows kernel's wavefronts take half a block each
    uint32_t tiled; // host side only: the split-K plan gives every 16 query vectors their own workgroups
    uint32_t whole_on_eight; // host side only: the split-K plan leaves every item whole on eight wavefronts
    uint32_t parts; // host side only: items are left whole in parts of channels: how many (attn_whole_f16.hip), or the channel
                    // tiles of one (attn_parts_halves.hip)
    uint32_t scale_scores; // host side only: AttnParams::scale_scores of a step in parts at head_dim 128
    uint32_t tile_sets;  // host side only: the tiles kernel's plan, sets of 16 query vectors a tile
    uint32_t tile_waves; // and wavefronts a workgroup
    uint32_t tile_exact; // and whether the softmax keeps the exact running maximum
    float plan_cost;     // host side only: what the block kernel's planner expects of its plan, us without the launch
    uint64_t partial_limit;  // host side only: bytes of partials the block kernel's plan may take (0 = any)
    AttnItem item[kMaxBatchItems];
};
// The kernel argument form of AttnBatch, sized to the batch: kernel arguments are
// expensive to read on this GPU (a 2.6 KB argument block costs about a microsecond per
// launch, a scan through 40-byte items several), so small batches get a small block.
//
// A workgroup finds its item in one trip to memory: every lane reads an item, the lanes compare side by side, and
// the fields come out of the lane that has it. Argument lines are cold at every launch and a trip to one costs 0.3 to 0.5 us;
// a walk over the items' first indices with the item's fields behind it was one trip an item and two more. One row of
// each slot, 32 Q / 4 KV heads, us a layer of attention and merge, walk -> this: 2 slots at 2,000 positions 8.2 -> 7.7, 8 at
// 500 9.0 -> 8.0, 16 of up to 1,000 12.0 -> 10.6, 32 at 300 10.7 -> 8.8, 16 of up to 16,384 58.5 -> 57.1; four slots of seven
// rows at 8,192 24.4 -> 23.7; f32, 8 KV heads, 6 slots at 900 16.5 -> 15.4.
template <int N>
struct AttnBatchT {
    uint32_t n;
    uint32_t total_blocks;
    uint32_t rows_per_block;
    uint32_t base_row;  // q_row0 of item 0
    AttnItem item[N];   // (those beyond n hold nothing)

    explicit AttnBatchT(const AttnBatch &b)
        : n(b.n), total_blocks(b.total_blocks), rows_per_block(b.rows_per_block),
          base_row(b.n ? b.item[0].q_row0 : 0) {
        for (uint32_t i = 0; i < b.n; ++i) item[i] = b.item[i];
    }
    // The item of a workgroup, or of a row of the batch: the last that does not begin beyond it. All lanes of the
    // wavefront ask together.
    __device__ __forceinline__ AttnItem of_block(uint32_t block) const {
        return fetch([=](const AttnItem &x) { return block >= x.block0; });
    }
    __device__ __forceinline__ AttnItem of_row(uint32_t row) const {
        const uint32_t at = base_row + row;
        return fetch([=](const AttnItem &x) { return at >= x.q_row0; });
    }

private:
    template <typename F>
    __device__ __forceinline__ AttnItem fetch(F begun) const {
        if constexpr (N == 1) {
            return item[0];
        } else {
            static_assert(N <= 64 && (N & (N - 1)) == 0, "an item a lane");
            const uint32_t lane = __lane_id() % N;
            const AttnItem mine = item[lane];
            const uint64_t mask = __builtin_amdgcn_ballot_w64(lane < n && begun(mine)) & (N == 64 ? ~0ull : (1ull << N) - 1);
            const uint32_t at = uint32_t(__builtin_popcountll(mask)) - 1u;
            AttnItem it;
#define ITAK_FIELD(f) it.f = __builtin_amdgcn_readlane(mine.f, at)
            ITAK_FIELD(slot), ITAK_FIELD(rows), ITAK_FIELD(pos0), ITAK_FIELD(q_row0), ITAK_FIELD(kv_len), ITAK_FIELD(splits);
            ITAK_FIELD(keys_per_split), ITAK_FIELD(block0), ITAK_FIELD(ws0), ITAK_FIELD(splits_magic), ITAK_FIELD(kv_lo);
#undef ITAK_FIELD
            return it;
        }
    }
};

// Runs CALL with `constexpr int N` set to the smallest of {1, 8, 64} that holds n items.
#define ITAK_DISPATCH_BATCH(n, CALL) \
    do {                              \
        if ((n) <= 1) {               \
            constexpr int N = 1;      \
            CALL;                     \
        } else if ((n) <= 8) {        \
            constexpr int N = 8;      \
            CALL;                     \
        } else {                      \
            constexpr int N = 64;     \
            CALL;                     \
        }                             \
    } while (0)

struct AttnParams {
    const void *layer_base;
    PoolGeom g;
    const float *q;
    float *out;
    const uint32_t *q_pos;  // optional explicit positions, [sum rows]
    float *ws;              // partials: (head_dim + 2) floats each
    // Fused append (split-K f16 kernel only): when set, the last `rows` positions of every
    // item are not in the cache yet; their K/V rows are read from here (row q_row0 + r,
    // [kv_heads*head_dim] f32 each), written to the cache by the kernel, and attended to.
    const float *k_new;
    const float *v_new;
    uint32_t q_heads;
    uint32_t group;         // q_heads / kv_heads
    uint32_t group_magic;   // ceil(2^16 / group): j / group == (j * magic) >> 16 for j < 64
    float scale;
    float softcap;
    uint32_t window;        // attention window of the layer (cache.rs:36-48); 0 = global
    uint32_t ring_blocks;   // 32-row blocks of the layer's storage ring; 0 = rows are positions
    // Split-K f16 kernel only: merge the splits inside the launch. `ws` is then the exchange
    // buffer (every word empty between launches) and item.ws0 counts its records; a consumer
    // gives up after spin_limit polls.
    uint32_t exchange;
    uint32_t spin_limit;
    // Block kernel only, unsplit causal launches: workgroups reach the device in runs of this
    // many (one per compute unit); every second run takes its units in reverse, so that the
    // two workgroups that share a compute unit are a long row tile and a short one. 0 = off.
    uint32_t fold_units;
    // The step's keys and values, over all layers of the pool, are more than the last-level cache
    // holds (so the next step will not find them there): kernels that read each row once may ask
    // for them with the streaming hint.
    uint32_t kv_streams;
    // Whole steps by channels (attn_whole_f16.hip) only: the queries are rounded to f16 as they are, and the scale goes
    // to the scores. Else the queries are rounded with the scale on.
    uint32_t scale_scores;
};
// What the reference's model does around the step (muse-glimmer/src/model.rs:445-464),
// folded into the step's own launches instead of running as launches of their own. `gate`
// (out *= sigmoid(gate), cpu.rs:657-673) is applied by whichever kernel writes the final
// output; `prep_on` makes the split-K kernel norm and rotate the raw Q rows and new K rows it
// reads (its 16-vector variants only). A separate kernel argument, so that launches without
// any of it carry and fetch nothing more.
struct FoldedParams {
    const float *gate;          // [sum rows][q_heads*head_dim] or null
    uint32_t prep_on;
    uint32_t prep_interleaved;  // 1: pairs (2i, 2i+1); 0: pairs (i, i + prep_rot/2)
    uint32_t prep_rot;          // rotary_dim; 0 = no rotation
    float prep_eps;
    const float *prep_q_weight; // [head_dim] or null: no norm
    const float *prep_k_weight;
    double prep_freq_step;      // pair i turns at position * 2^(i * prep_freq_step) radians,
    const double *prep_freq;    // which is prep_freq[i] where the host could make the table
};
// sigmoid for the writers of f16-KV attention output, whose bar is 2e-3: one exponential
// and one reciprocal instruction, a few ulp, the same limits at both ends (0 and 1) as the
// reference's two-branch form (cpu.rs:162-169).
__device__ __forceinline__ float sigmoid_fast(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}
// sigmoid as the reference writes it (cpu.rs:162-169).
__device__ __forceinline__ float sigmoid_ref(float x) {
    if (x >= 0.0f) return 1.0f / (1.0f + expf(-x));
    const float e = expf(x);
    return e / (1.0f + e);
}
// The oldest position a query at `pos` sees (attention.rs:77-85 and the view's oldest row).
__host__ __device__ inline uint32_t lowest_visible(uint32_t pos, uint32_t window, uint32_t kv_lo) {
    const uint32_t lo = (window != 0 && pos + 1 > window) ? pos + 1 - window : 0;
    return lo > kv_lo ? lo : kv_lo;
}

// Generic VALU path: f32 or f16 storage, any head_dim <= 256, group <= 64. Partials are in
// natural-log domain (combine with base2 = 0).
hipError_t launch_attn_generic(int elem_f16, const AttnParams &p, const AttnBatch &b,
                               uint32_t total_partials, hipStream_t stream);
// Query rows one workgroup of the generic kernel carries (0 = shape not supported).
uint32_t attn_generic_rows_per_block(uint32_t group, uint32_t head_dim);
// Keys per tile of the generic kernel for a head_dim.
uint32_t attn_generic_tile(uint32_t head_dim);

// MFMA split-K path: f16 pools with blocked value planes, head_dim 128, rows*group <= 64.
// Partials are in log2 domain (combine with base2 = 1).
bool attn_splitk_f16_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows);
// (`prepares`: the launch prepares Q and the new K rows itself.)
uint32_t attn_splitk_f16_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, bool prepares = false, bool may_tile = false,
                              bool may_part = false);
// After attn_splitk_f16_plan: whether the batch can merge its splits inside the split-K launch
// (AttnParams::exchange). Returns the 64-bit words the exchange buffer must hold and re-bases
// the items' ws0 on it, or 0 (items untouched) when the batch keeps the merge launch.
uint64_t attn_splitk_f16_plan_exchange(const PoolGeom &g, AttnBatch &b, uint32_t q_heads);
// Sets `count` 64-bit words to `value` (the exchange buffer's empty pattern, at set-up).
hipError_t launch_fill_words(unsigned long long *dst, uint64_t count, unsigned long long value,
                             hipStream_t stream);
constexpr unsigned long long kExchangeEmptyWord = 0xffffffffffffffffull;
// `folded` with prep_on set selects the variants that prepare Q and the new K rows themselves
// and gate what they write (every item must then be a 16-vector step); otherwise it is ignored.
// `q_two_halves`: the queries enter the score products as f16 hi + f16 lo (two products per
// score tile), so that their rounding to f16 leaves the scores (ITAK_POOL_Q_TWO_HALVES).
hipError_t launch_attn_splitk_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  uint32_t max_rows, hipStream_t stream,
                                  const FoldedParams *folded = nullptr, bool q_two_halves = false);
// The two-halves instantiations (attn_splitk_f16_qlo.hip) and the variant a batch takes.
hipError_t launch_attn_splitk_f16_qlo(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                      hipStream_t stream, const FoldedParams *folded);
int attn_splitk_f16_variant(const PoolGeom &g, const AttnBatch &b, uint32_t group);
// ---- the split merge on a unit's compute die (attn_splitk_f16_die.hip) ---------------------
// The device's workgroups are dealt round-robin over its eight compute dies, each with an L2 of
// its own. A launch planned for it puts every split of a unit = (item, KV head, part of the
// query vectors) on one die; the unit's last workgroup to finish merges the partials out of
// that die's L2, so there is neither a merge launch nor a wait.
constexpr uint32_t kDieCount = 8;
constexpr uint32_t kDieTicketStride = 32;  // words from one unit's ticket to the next: a cache line each
constexpr uint32_t kDieMaxUnits = 1024;
constexpr uint64_t kDieTicketBytes = uint64_t(kDieMaxUnits) * kDieTicketStride * 4;
struct DieMap {
    uint32_t *tickets;  // kDieMaxUnits words kDieTicketStride apart, zero whenever no launch runs
    uint32_t *faults;   // workgroups that found themselves on another die than their index names
    const float *gate;  // merged rows are multiplied by sigmoid(gate) as they are written, or null
    uint32_t shift;     // log2(heads a bin's dies share out): die = bin << shift | KV head
    uint32_t pad;
    uint32_t bin_first[kDieCount + 1];  // items of bin i: [bin_first[i], bin_first[i + 1])
    uint32_t bin_count[kDieCount];      // workgroups of a die of bin i
};
// True when the current device deals workgroup i to compute die i % 8 (probed once per device:
// a small launch whose workgroups report the hardware's die number).
bool die_layout_ok(int device);
// Plans `b` (slot, rows, pos0, q_row0, kv_len, kv_lo set) for the die-local merge: `out` gets
// the items in bin order with splits, keys_per_split, block0 (first index on the die), ws0 and
// the unit's first ticket (in splits_magic); `map` the bins. Returns the partials the launch
// writes, 0 when the batch is better served by the ordinary plan (too few or too uneven units,
// a KV head count that does not deal out over eight dies, nothing to split).
uint32_t attn_splitk_f16_plan_die(const PoolGeom &g, const AttnBatch &b, uint32_t q_heads,
                                  AttnBatch &out, DieMap &map);
hipError_t launch_attn_splitk_f16_die(const AttnParams &p, const AttnBatch &b, const DieMap &map,
                                      uint32_t total_partials, hipStream_t stream,
                                      const FoldedParams *folded = nullptr);
// The latency-shaped form of the same path for decode steps (attn_decode_f16.hip): every item
// one new row, at most one block per wavefront, splits merged inside the launch. `takes` is
// asked after the batch has been planned and AttnParams::exchange set.
bool attn_decode_f16_takes(const AttnParams &p, const AttnBatch &b);
// Workgroups of that kernel the device holds at once (the smallest figure over its
// instantiations, asked of the runtime once).
uint32_t attn_decode_f16_resident_groups();
// `prepares`: Q and the new K rows are prepared by the launch (not with q_two_halves or an exchange).
hipError_t launch_attn_decode_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  hipStream_t stream, bool q_two_halves = false, const FoldedParams *prepares = nullptr);
// Whole one-row steps by channels (attn_whole_f16.hip): AttnBatch::parts is 2, 4 or 8.
constexpr uint32_t kWholeMostBlocks = 24;
hipError_t launch_attn_whole_f16(const AttnParams &p, const AttnBatch &b, hipStream_t stream, const FoldedParams *prepares);
// f32 MFMA split-K path: f32 pools (row-major planes), head_dim 128, rows*group <= 16, implied
// query positions. Partials are in log2 domain (combine with base2 = 1).
bool attn_splitk_f32_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows);
// (`groups_per_cu` workgroups of four wavefronts share a compute unit; `partial_bytes`: the workspace of a call
// that may not grow it, 0 = any; `may_part` = false: no steps by channels, attn_parts_halves.hip.)
uint32_t attn_splitk_f32_plan(const PoolGeom &g, int elem_f16, AttnBatch &b, uint32_t q_heads, uint32_t groups_per_cu,
                              uint64_t partial_bytes, bool may_part);
hipError_t launch_attn_splitk_f32(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  hipStream_t stream);
// f32-arithmetic MFMA split-K path for the other shapes (attn_splitk_any.hip): f16 and f32 pools,
// any head_dim <= 256 that is a multiple of four, any group, implied query positions, tensors
// 16-byte aligned. Planned by attn_splitk_f32_plan; partials are in log2 domain.
bool attn_splitk_any_supports(const PoolGeom &g, uint32_t group, uint32_t max_rows);
// Workgroups of that kernel a compute unit holds.
uint32_t attn_splitk_any_groups_per_cu(const PoolGeom &g);
// True when such a launch also appends the step's rows (k_new / v_new in its parameters); launches of
// the f32 kernel always do.
bool attn_splitk_any_appends(const PoolGeom &g, int elem_f16, uint32_t group, uint32_t max_rows);
// One-row steps by channels on blocked f16 planes at other head dims (attn_parts_halves.hip); `plan` = whether it took the
// batch, and its partials.
bool attn_parts_halves_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, uint32_t *partials);
hipError_t launch_attn_parts_halves(const AttnParams &p, const AttnBatch &b, uint32_t total_partials, hipStream_t stream);
hipError_t launch_attn_splitk_any(int elem_f16, const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                  hipStream_t stream);
// MFMA block path (speculative blocks and prefill chunks): same pools, any number of rows,
// group dividing 16; K/V staged through LDS, split over the context when the launch would
// otherwise not fill the device. Partials are in log2 domain (combine with base2 = 1).
bool attn_prefill_f16_supports(const PoolGeom &g, uint32_t group);
uint32_t attn_prefill_f16_plan(const PoolGeom &g, AttnBatch &b, uint32_t group, uint32_t q_heads,
                               uint32_t window, bool appends = false);
// True when a launch of the block kernel over items of at most `most_rows` rows and
// `most_blocks` key blocks appends the items' rows itself (k_new / v_new in its parameters).
bool attn_prefill_f16_appends(const PoolGeom &g, uint32_t group, uint32_t most_rows,
                              uint32_t most_blocks);
hipError_t launch_attn_prefill_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                   hipStream_t stream);
// The same at head dims 64, 96 and 256 (instantiated in a file of their own); `one` = the
// one-tile form, as launch_attn_prefill_f16 decides it.
// The two-halves form (head_dim 128, two tiles, no rows brought along).
hipError_t launch_attn_prefill_f16_qlo(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                       hipStream_t stream);
hipError_t launch_attn_prefill_f16_dims(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                                        bool one, hipStream_t stream);
// Tiles of 16 or 32 query vectors whose wavefronts split the keys (attn_tiles_f16.hip): blocks of some
// rows on the same pools at head_dim 128, new rows brought along or appended before. The batch's plan
// says which form; `gate` multiplies the rows of items with one split.
struct TilesPlan {
    uint32_t sets = 0;   // of 16 query vectors a tile; 0 = the launch is another kernel's
    uint32_t waves = 0;
    uint32_t run = 0;    // blocks a split walks at most
    bool appends = false; // the launch brings the step's rows along
    bool exact = false;   // the softmax keeps the exact running maximum
};
bool attn_tiles_f16_supports(const PoolGeom &g, uint32_t group, uint32_t most_rows);
// The cheapest form for a batch (slot, rows, pos0, kv_len, kv_lo set) that costs less than `below` us, and its cost
// (`below` and the plan as it was when there is none). `brings_rows`: the
// step's rows are not in the cache yet (appended by the launch where the form can, else before it); `few_rows`: a
// step the split-K kernel takes as well.
float attn_tiles_f16_choose(const PoolGeom &g, const AttnBatch &b, uint32_t q_heads, uint32_t window, bool brings_rows,
                            bool few_rows, uint64_t partial_limit, float below, TilesPlan &plan);
uint32_t attn_tiles_f16_plan(const PoolGeom &g, AttnBatch &b, uint32_t q_heads, const TilesPlan &plan);
hipError_t launch_attn_tiles_f16(const AttnParams &p, const AttnBatch &b, uint32_t total_partials, const float *gate,
                                 hipStream_t stream);
// Merge of split partials; total_rows = query rows of the batch. With `gate` the merged rows
// are multiplied by sigmoid(gate) as they are written (items with one split are not touched:
// their writer was the attention kernel).
hipError_t launch_attn_combine(const AttnParams &p, const AttnBatch &b, uint32_t total_partials,
                               uint32_t total_rows, int base2, hipStream_t stream,
                               const float *gate = nullptr);

}  // namespace itak
