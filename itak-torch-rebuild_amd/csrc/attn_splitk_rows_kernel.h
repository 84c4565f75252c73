// The split-K attention kernel over row-major planes: f32 pools (the reference's own storage type)
// and f16 pools whose head_dim is no multiple of 16. Products on v_mfma_f32_16x16x4_f32 (f32 in, f32
// out: the 1e-5 bar of f32 pools holds), K and V read straight from their planes, no LDS in the
// loop. Instantiated in attn_splitk_f32.hip (f32, head_dim 64 and 128) and attn_splitk_any.hip.
//
// One workgroup of four or eight wavefronts owns (item, KV head, tile of 16 query vectors, split = a run of
// 32-key blocks), a query vector being one row of one Q head of the group; a block of more than 16
// vectors is several tiles, each walking the keys its own rows see (tiles of later rows first: they
// have the longest runs). Each wavefront walks its own blocks with a private online softmax, the
// wavefronts merge once through LDS. The MFMA takes one float per lane and operand: A[i][k] from lane
// i + 16k, B[k][j] from lane j + 16k, and returns rows 4g .. 4g+3 of column j to lane j + 16g. A dot
// product does not care in which order its terms are taken, so the channels (for K.Q^T) and the
// keys (for V^T.P^T) are assigned to the MFMA's k index in whatever order lets every lane fetch four
// consecutive channels:
//
//   S^T = K . Q^T   per 16-key tile t, steps (s, e): lane (i, g) supplies K[key 16t + i][channel
//                   16s + 4g + e], i.e. the piece at channels 16s + 4g of its key row covers the four
//                   e of a step group; Q^T is held the same way. Lane (j, g) receives the scores of
//                   keys 16t + 4g + r, r = 0..3.
//   O^T += V^T . P^T  per tile t and r = 0..3 the k index g stands for key 16t + 4g + r, whose
//                   probability is exactly what lane (j, g) holds in score register r: P needs no
//                   shuffle. Output tile (h, e) row i is channel 64h + 4i + e, so lane (i, g) fetches
//                   the piece at channels 64h + 4i of value row 16t + 4g + r.
//
// A launch of one block per wavefront is a chain of latencies, so the order of its requests counts:
// raw queries, then the first block's keys and values, and only then anything that waits; a later
// block's keys are asked for as soon as the scores have used up the operands, its values behind the
// products. (With Q converted before the first key was asked for, and with the row-by-row treatment
// of values that are not finite inside the loop, which cost a multi-row launch its second workgroup
// per compute unit, 9 rows of 32 Q / 4 KV heads at context 3,000 took 16.8 us.)
//
// gqa_attention never reads the key or value row of a position a query does not see
// (crates/attention/src/attention.rs:160-173), but the rows of a tile share the value operand here,
// and a masked key's zero weight times a value that is not finite is NaN. A wavefront whose sums
// come out not finite walks its keys again, query row by query row, with the keys a row does not see
// cleared: rolled loops, cold and small.
//
// Semantics: gqa_attention in crates/attention/src/attention.rs:104-215, softcap as
// crates/torch-math/src/logits.rs:26-37. Partials are in the log2 domain.
#pragma once

#include "internal.h"
#include "mfma_common.h"
#include "split_exchange.h"

namespace itak {

namespace {


__device__ __forceinline__ float lanes4_max(float v) {  // over lanes l, l^16, l^32, l^48
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float lanes4_sum(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// x = h[0] + h[1] + h[2] up to 2^-33 of the largest x the halves hold. A half that is not finite
// has nothing left to say.
__device__ __forceinline__ void split3(float x, _Float16 &a, _Float16 &b, _Float16 &c) {
    a = static_cast<_Float16>(x);
    const float r = x - float(a);
    b = static_cast<_Float16>(r);
    c = static_cast<_Float16>(r - float(b));
}

// Weights carry this many powers of two (so that their third halves are no subnormals); sums and
// outputs carry them too, and lose them in the division.
constexpr float kWeightShift = 15.0f;

// Four channels of a row. K/V rows that one workgroup alone reads (a step of one tile of vectors
// per KV head: decode rows, short blocks) are read with the streaming hint, so that they do not
// displace the kernel's code, arguments and split partials in L2 (decode at context 4096 13.6 ->
// 12.65 us per layer, the ragged batch 86.1 -> 81.5). Rows that several tiles' workgroups read keep
// the plain load: with the hint a 2048-row chunk took 4.4 ms instead of 3.3.
template <typename T>
struct Piece4;
template <>
struct Piece4<float> {
    floatx4 v;
    template <bool STREAM>
    __device__ __forceinline__ void load(const float *p) {
        v = STREAM ? __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(p)) : *reinterpret_cast<const floatx4 *>(p);
    }
    __device__ __forceinline__ float at(int e) const { return v[e]; }
    __device__ __forceinline__ void clear() { v = floatx4{0.f, 0.f, 0.f, 0.f}; }
    static __device__ __forceinline__ float one(const float *p) { return *p; }
    static __device__ __forceinline__ void store(float *p, floatx4 x) { *reinterpret_cast<floatx4 *>(p) = x; }
};
template <>
struct Piece4<uint16_t> {
    half4 v;
    template <bool STREAM>
    __device__ __forceinline__ void load(const uint16_t *p) {
        v = STREAM ? __builtin_nontemporal_load(reinterpret_cast<const half4 *>(p)) : *reinterpret_cast<const half4 *>(p);
    }
    __device__ __forceinline__ float at(int e) const { return float(v[e]); }
    __device__ __forceinline__ void clear() { v = half4{}; }
    static __device__ __forceinline__ float one(const uint16_t *p) { return float(__builtin_bit_cast(_Float16, *p)); }
    static __device__ __forceinline__ void store(uint16_t *p, floatx4 x) {
        uint2 h = {f32_to_f16_bits(x[0]) | uint32_t(f32_to_f16_bits(x[1])) << 16,
                   f32_to_f16_bits(x[2]) | uint32_t(f32_to_f16_bits(x[3])) << 16};
        *reinterpret_cast<uint2 *>(p) = h;
    }
};

// DP: head_dim rounded up to a multiple of 64 (pieces beyond head_dim are read from the row's last
// and taken as zero); EXACT: it is head_dim. TT: 16-key tiles whose rows are in registers at a time
// (1 where two would not fit). W: wavefronts. HALF: they take half a block each, in turn.
template <typename T, int DP, bool EXACT, int TT, bool STREAM, int W, bool kHalf, int N>
__global__ __launch_bounds__(W * 64, DP <= 128 && W == 4 ? 2 : 1) void attn_splitk_rows_kernel(AttnParams p, AttnBatchT<N> b,
                                                                                             uint32_t total_partials) {
    static_assert(!kHalf || TT == 1, "half a block is one tile");
    constexpr int kTiles = DP / 16;  // output tiles (h, e)
    constexpr int kS = DP / 16;      // pieces of a key row per lane group
    constexpr int kH = DP / 64;      // pieces of a value row per lane
    __shared__ float sm_m[W][16], sm_l[W][16];
    __shared__ floatx4 sm_q[DP * 4];
    // [wave][tile][row of the lane][lane]: written and read a float a lane without bank conflicts (with the
    // lane's four rows side by side the merge's reads were four-way conflicts, 0.4 us of a one-row step).
    __shared__ float sm_o[W][kTiles][4][64];

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = tid >> 6, lane = tid & 63;
    const uint32_t g = lane >> 4, jl = lane & 15;
    const uint32_t D = EXACT ? DP : p.g.head_dim;

    const AttnItem item = b.of_block(blockIdx.x);
    const uint32_t local = blockIdx.x - item.block0;
    const uint32_t unit = local / item.splits, split = local % item.splits;
    const uint32_t group = p.group, nvec = item.rows * group;
    const uint32_t vtiles = (nvec + 15) / 16;
    const uint32_t kv_head = unit % p.g.kv_heads, vtile = vtiles - 1 - unit / p.g.kv_heads;
    // The rows this tile's vectors belong to bound the keys it walks.
    const uint32_t row_first = (vtile * 16) / group;
    const uint32_t row_last = min(item.rows - 1, (vtile * 16 + 15) / group);

    T *kplane = static_cast<T *>(const_cast<void *>(p.layer_base)) + item.slot * p.g.slot_stride + kv_head * p.g.head_stride;
    T *vplane = kplane + p.g.side_stride;

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
    // [tile_lo, tile_hi): the positions some row of this tile sees.
    const uint32_t tile_lo = lowest_visible(item.pos0 + row_first, window, kv_lo);
    const uint32_t tile_hi = min(item.pos0 + row_last + 1, item.kv_len);
    const float softcap = p.softcap;
    const float inv_cap = softcap > 0.0f ? 1.0f / softcap : 0.0f;
    const float qscale = softcap > 0.0f ? p.scale : p.scale * kLog2e;
    const float *qp = p.q + (uint64_t(item.q_row0 + row) * p.q_heads + head) * D;

    // Channels of a lane's pieces. Only those of the last 64 can lie beyond head_dim.
    auto key_piece = [&](int s) { return EXACT || 16 * (s + 1) <= DP - 64 ? 16u * s + 4 * g : min(16u * s + 4 * g, D - 4); };
    auto value_piece = [&](int h) { return EXACT || h + 1 < kH ? 64u * h + 4 * jl : min(64u * h + 4 * jl, D - 4); };

    // Q^T as B operands: step (s, e) takes channel 16s + 4g + e of vector jl. The tile's vectors are read
    // once and handed round through LDS, piece (s, g, vector) at (4s + g) * 16 + vector: read by every
    // wavefront they are a third of what a compute unit's load path moves for a block.
    constexpr int kQ = (DP * 4 + W * 64 - 1) / (W * 64);  // pieces a thread stages
    floatx4 q_raw[kQ];
#pragma unroll
    for (int u = 0; u < kQ; ++u) {
        const uint32_t f = min(tid + u * W * 64, DP * 4u - 1), c4 = (f / 16) * 4, vj = min(vtile * 16 + f % 16, nvec - 1);
        const uint32_t r = vj / group, hd = kv_head * group + vj - r * group;
        q_raw[u] = *reinterpret_cast<const floatx4 *>(p.q + (uint64_t(item.q_row0 + r) * p.q_heads + hd) * D +
                                                      (EXACT ? c4 : min(c4, D - 4)));
    }

    // A step of the walk: TT tiles of block kb, from tile t0.
    Piece4<T> k[TT][kS], v[TT][4][kH];
    // Fused append (p.k_new set). f32 rows: whoever reads a new position reads it where the caller left
    // it, so nothing waits for a store, and a row is copied to the planes at the end by the workgroups of
    // the tile its first vector is in, its splits taking the pieces in turn. (Not by the last tile's, which
    // walk every block of a global layer: on a windowed one none of them walks the rows below that tile's
    // window, and a cut brings those back into view. A chunk's stores are also spread over the launch
    // instead of kv_heads * splits workgroups: 32 Q / 4 KV heads, head_dim 128, 256 rows from an empty
    // cache 24.9 -> 14.9 us a layer, 1,024 139 -> 111.) (Every step takes its rows' addresses through the same selects: as a path of its own, which only the last block's wavefront
    // ran, cold, it cost a one-row launch 0.8 us.) f16 rows: the wavefront that owns
    // a block stores the new rows in it and waits for the stores before it reads the block (where several
    // tiles' workgroups walk the block, each stores the same rows and reads its own).
    constexpr bool kInPlace = sizeof(T) == 4;
    const bool fused = p.k_new != nullptr;
    const uint32_t fresh_from = kInPlace && fused ? item.pos0 : 0xffffffffu;
    const uint32_t new_stride = p.g.kv_heads * D;
    const uint64_t new_at = uint64_t(item.q_row0) * new_stride + kv_head * D;
    // Row i of the step: its storage row, and where its data is. Rows past the stored length are read
    // from the last stored row instead (the plane may end there) and masked.
    auto step_pos = [&](uint32_t kb, uint32_t t0, uint32_t i) { return min(kb * kBlockKeys + 16 * t0 + i, item.kv_len - 1); };
    auto step_row = [&](uint32_t kb, uint32_t t0, uint32_t i) {
        return (ring_blocks ? kb % ring_blocks : kb) * kBlockKeys + step_pos(kb, t0, i) - kb * kBlockKeys;
    };
    auto row_at = [&](const T *plane, const float *fresh, uint32_t kb, uint32_t t0, uint32_t i) -> const T * {
        if constexpr (kInPlace) {
            const uint32_t pos = step_pos(kb, t0, i);
            const bool is_new = pos >= fresh_from;
            const uint32_t row = is_new ? pos - item.pos0 : step_row(kb, t0, i);
            return (is_new ? fresh + new_at : plane) + uint64_t(row) * (is_new ? new_stride : D);
        } else {
            return plane + uint64_t(step_row(kb, t0, i)) * D;
        }
    };
    auto load_keys = [&](uint32_t kb, uint32_t t0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const T *kr = row_at(kplane, p.k_new, kb, t0, 16 * t + jl);
#pragma unroll
            for (int s = 0; s < kS; ++s) k[t][s].template load<STREAM>(kr + key_piece(s));
            if (kInPlace) __builtin_amdgcn_sched_barrier(0);  // (all rows' addresses at once would not fit)
        }
    };
    auto load_values = [&](uint32_t kb, uint32_t t0) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const T *vr = row_at(vplane, p.v_new, kb, t0, 16 * t + 4 * g + r);
#pragma unroll
                for (int h = 0; h < kH; ++h) v[t][r][h].template load<STREAM>(vr + value_piece(h));
                if (kInPlace) __builtin_amdgcn_sched_barrier(0);
            }
    };
    // The rows this workgroup copies (see above). A thread's first piece is asked for now and stored at
    // the end.
    const uint32_t own_from = row_first + (row_first * group < vtile * 16 ? 1 : 0), own_to = row_last + 1;
    const uint32_t quads = D / 4;
    const uint32_t own_base = (item.splits - 1 - split) * (W * 64);  // (the last split's run is the shortest)
    const uint32_t own_rows = kInPlace && fused && own_to > own_from ? own_to - own_from : 0;
    const uint32_t own_pieces = own_base < own_rows * 2 * quads ? own_rows * 2 * quads : 0;
    const uint32_t own_first = own_base + tid;
    auto own_piece = [&](uint32_t f, const float *&src, T *&dst) {
        const uint32_t r = own_from + f / (2 * quads), rest = f % (2 * quads), side = rest >= quads ? 1 : 0;
        const uint32_t pos = item.pos0 + r, c4 = (rest - side * quads) * 4;
        src = (side ? p.v_new : p.k_new) + new_at + uint64_t(r) * new_stride + c4;
        dst = (side ? vplane : kplane) + uint64_t(ring_blocks ? pos % (ring_blocks * kBlockKeys) : pos) * D + c4;
    };
    floatx4 own = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    if (own_first < own_pieces) {
        const float *src;
        T *dst;
        own_piece(own_first, src, dst);
        own = *reinterpret_cast<const floatx4 *>(src);
    }
    auto store_own = [&] {
        for (uint32_t f = own_first; f < own_pieces; f += item.splits * (W * 64)) {
            const float *src;
            T *dst;
            own_piece(f, src, dst);
            if (f != own_first) own = *reinterpret_cast<const floatx4 *>(src);
            Piece4<T>::store(dst, own);
        }
    };
    auto append_rows = [&](uint32_t kb, uint32_t t0) {
        if constexpr (!kInPlace) {
        const uint32_t key0 = kb * kBlockKeys + (kHalf ? 16 * t0 : 0), keys = kHalf ? 16 : kBlockKeys;
        if (!fused || key0 + keys <= item.pos0 || key0 >= item.pos0 + item.rows) return;
        const uint32_t from = key0 > item.pos0 ? key0 - item.pos0 : 0;
        const uint32_t to = min(item.rows, key0 + keys - item.pos0), quads = D / 4;
        for (uint32_t f = lane; f < (to - from) * 2 * quads; f += 64) {
            const uint32_t r = from + f / (2 * quads), rest = f % (2 * quads);
            const uint32_t side = rest >= quads ? 1 : 0, c4 = (rest - side * quads) * 4;
            const floatx4 y = *reinterpret_cast<const floatx4 *>(
                (side ? p.v_new : p.k_new) + (uint64_t(item.q_row0 + r) * p.g.kv_heads + kv_head) * D + c4);
            const uint32_t srow = (ring_blocks ? kb % ring_blocks : kb) * kBlockKeys + (item.pos0 + r) % kBlockKeys;
            Piece4<T>::store((side ? vplane : kplane) + uint64_t(srow) * D + c4, y);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores have been acknowledged
        }
    };
    auto advance = [&](uint32_t &kb, uint32_t &t0) {
        if constexpr (kHalf) {
            kb += W / 2;
        } else {
            t0 += TT;
            if (t0 == 2) {
                t0 = 0;
                kb += W;
            }
        }
    };
    uint32_t kb = kb_begin + (kHalf ? wave / 2 : wave), t0 = kHalf ? wave & 1 : 0;
    if (kb < kb_end) append_rows(kb, t0);
    {
        // (A wavefront without a block loads one and ignores it: behind a branch the wait for the queries
        // would be a wait for every load, and the barrier below the slowest wavefront's.)
        const uint32_t some = min(kb, (item.kv_len - 1) / kBlockKeys);
        load_keys(some, t0);
        load_values(some, t0);
    }
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int u = 0; u < kQ; ++u) {
        const uint32_t f = tid + u * W * 64;
        floatx4 x = q_raw[u] * qscale;
        if (vtile * 16 + f % 16 >= nvec || (!EXACT && (f / 16) * 4 >= D)) x = floatx4{0.f, 0.f, 0.f, 0.f};
        if (f < DP * 4u) sm_q[f] = x;
    }
    lds_barrier();
    floatx4 q[kS];
#pragma unroll
    for (int s = 0; s < kS; ++s) q[s] = sm_q[s * 64 + lane];

    float m_run = -INFINITY, l_run = 0.0f;
    floatx4 o[kTiles];
#pragma unroll
    for (int c = 0; c < kTiles; ++c) o[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // What both walks do with a step's scores: cap, mask, running maximum and sum; sc becomes the
    // weights, and the return value what the earlier steps' outputs are worth now.
    auto weigh = [&](uint32_t key0, float (&sc)[TT][4]) -> float {
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t kp = key0 + 16 * t + 4 * g + r;
                float x = sc[t][r];
                if (softcap > 0.0f) x = softcap_log2(x, softcap, inv_cap);
                if (kp > colpos || kp < collo) x = -INFINITY;
                sc[t][r] = x;
                mx = fmaxf(mx, x);
            }
        mx = lanes4_max(mx);
        const float m_new = fmaxf(m_run, mx);
        const bool dead = m_new == -INFINITY;
        const float alpha = (dead || m_run == -INFINITY) ? (dead ? 1.0f : 0.0f) : fast_exp2(m_run - m_new);
        float sum = 0.0f;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (Nothing finite in sight so far: -inf weighs zero against a reference of zero,
                // and a NaN score, which the maximum passes over as the reference's comparison
                // does, stays NaN and takes the row with it.)
                const float pe = fast_exp2(sc[t][r] - (dead ? 0.0f : m_new));
                sc[t][r] = pe;
                sum += pe;
            }
        l_run = l_run * alpha + sum;
        m_run = m_new;
        return alpha;
    };

    while (kb < kb_end) {
        const uint32_t key0 = kb * kBlockKeys + 16 * t0;
        uint32_t next_kb = kb, next_t0 = t0;
        advance(next_kb, next_t0);
        float sc[TT][4];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                // (Only the last four pieces can lie beyond head_dim, and then not in all lanes.)
                if (!EXACT && (s + 1) * 16 > DP - 64 && 16u * s + 4 * g >= D) k[t][s].clear();
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][s].at(e), q[s][e], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[t][r] = acc[r];
        }
        if (next_kb < kb_end) {
            if (kHalf || next_t0 == 0) append_rows(next_kb, next_t0);
            load_keys(next_kb, next_t0);
        }
        const float alpha = weigh(key0, sc);
        // A row no query of the tile sees (past the stored length or the tile's last row, or older
        // than its oldest window on a ring) may hold anything, stale data or a value that is not
        // finite: keep it out of P.V even as 0*x.
        if (key0 + 16 * TT > tile_hi || key0 < tile_lo) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t kp = key0 + 16 * t + 4 * g + r;
                    if (kp >= tile_hi || kp < tile_lo) {
#pragma unroll
                        for (int h = 0; h < kH; ++h) v[t][r][h].clear();
                    }
                }
        }
#pragma unroll
        for (int c = 0; c < kTiles; ++c) o[c] *= alpha;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < kTiles; ++c)
                    o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][r][c / 4].at(c % 4), sc[t][r], o[c], 0, 0, 0);
        if (next_kb < kb_end) load_values(next_kb, next_t0);
        kb = next_kb;
        t0 = next_t0;
    }

    float all = l_run;
#pragma unroll
    for (int c = 0; c < kTiles; ++c) {
        // (Output rows beyond head_dim hold whatever the clamped pieces gave.)
        all += (o[c][0] + o[c][1]) + (o[c][2] + o[c][3]);
#pragma unroll
        for (int r = 0; r < 4; ++r) sm_o[wave][c][r][lane] = o[c][r];
    }
    if (__builtin_amdgcn_ballot_w64(!(fabsf(all) < INFINITY)) != 0) {
#pragma unroll 1
        for (uint32_t c = 0; c < kTiles; ++c) {
            const uint32_t ch_out = min(64 * (c / 4) + 4 * jl + c % 4, D - 1);
            m_run = -INFINITY;
            l_run = 0.0f;
            floatx4 out = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (uint32_t sb = kb_begin + (kHalf ? wave / 2 : wave); sb < kb_end; sb += kHalf ? W / 2 : W)
#pragma unroll 1
                for (uint32_t st = kHalf ? wave & 1 : 0; st < 2; st += kHalf ? 2 : TT) {
                    const uint32_t key0 = sb * kBlockKeys + 16 * st;
                    floatx4 acc[TT] = {};
#pragma unroll 1
                    for (uint32_t ch = g; ch < D; ch += 4) {  // head_dim is a multiple of 4: every lane takes each turn
                        const float qv = jv < nvec ? qp[ch] * qscale : 0.0f;
#pragma unroll
                        for (int t = 0; t < TT; ++t)
                            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                Piece4<T>::one(row_at(kplane, p.k_new, sb, st, 16 * t + jl) + ch), qv, acc[t], 0, 0, 0);
                    }
                    float sc[TT][4];
#pragma unroll
                    for (int t = 0; t < TT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) sc[t][r] = acc[t][r];
                    out *= weigh(key0, sc);
                    float x[TT][4];
#pragma unroll
                    for (int t = 0; t < TT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            x[t][r] = Piece4<T>::one(row_at(vplane, p.v_new, sb, st, 16 * t + 4 * g + r) + ch_out);
#pragma unroll 1
                    for (uint32_t rr = row_first; rr <= row_last; ++rr) {
                        const uint32_t pos = min(item.pos0 + rr, item.kv_len - 1);
                        const uint32_t lo = lowest_visible(item.pos0 + rr, window, kv_lo);
                        floatx4 part = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int t = 0; t < TT; ++t)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const uint32_t kp = key0 + 16 * t + 4 * g + r;
                                part = __builtin_amdgcn_mfma_f32_16x16x4f32(kp <= pos && kp >= lo ? x[t][r] : 0.0f, sc[t][r], part,
                                                                            0, 0, 0);
                            }
                        if (row == rr) out += part;
                    }
                }
#pragma unroll
            for (int r = 0; r < 4; ++r) sm_o[wave][c][r][lane] = out[r];
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
    store_own();
    if (jv >= nvec) return;
    const bool final_out = item.splits == 1;
    const uint64_t ps = item.ws0 + (uint64_t(row) * p.q_heads + head) * item.splits + split;
    float *dst = final_out ? p.out + (uint64_t(item.q_row0 + row) * p.q_heads + head) * D : p.ws + ps * D;
    const float post = final_out ? 1.0f / L : 1.0f;
    // Tile (h, e), register rr = channel 64h + 16g + 4rr + e: wavefront w finishes register w % 4 of
    // every (of eight: every second) h.
    const uint32_t rr = wave % 4;
    for (int h = wave / 4; h < kH; h += W / 4) {
        const uint32_t ch = 64 * h + 16 * g + 4 * rr;
        floatx4 fin = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w)
#pragma unroll
            for (int e = 0; e < 4; ++e) fin[e] = fmaf(sm_o[w][4 * h + e][rr][lane], wgt[w], fin[e]);
        fin *= post;
        if (EXACT || ch < D) *reinterpret_cast<floatx4 *>(dst + ch) = fin;
    }
    if (!final_out && wave == 0 && g == 0)
        *reinterpret_cast<float2 *>(p.ws + uint64_t(total_partials) * D + ps * 2) = make_float2(M, L);
}

}  // namespace

}  // namespace itak
