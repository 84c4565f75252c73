// FNV-1a 64 (crates/itak-kv/src/hash.rs:24-31) of a long run of bytes in device memory.
//
// The hash is a chain, h = (h ^ byte) * p, one multiply per byte that waits for the last: a host
// core walks it at about 1.2 GB/s and no faster. Two facts about the chain take it apart:
//   - the xor touches only the low byte, so with l the low byte and t = l ^ byte, the step is
//     h' = (h + t - l) * p: once the low bytes along the chain are known it is affine in h, and a
//     run of n bytes started from h = l instead of h ends at (its own end) + (h - l) * p^n;
//   - the low bytes are a chain of their own, l' = (l ^ byte) * 0xb3 mod 256, in which bit k of a
//     value depends on bits 0..k before it alone, and flipping bit k of the start flips bit k of
//     the end and no lower one.
// So the low byte is found two bits at a time: a thread walks its 64 bytes from the two starts
// that differ in the lower of the two bits (both in one register, 16 bits each); how the pair of
// bits is carried over the run is then four bits of table (the upper bit of the start is just
// xored through), tables compose, and a scan over threads, workgroups and the whole run gives
// every thread the pair it starts from. After four rounds every thread knows the byte, walks its
// 64 bytes once more in 64 bits, and a weighted sum joins the runs.
//
// Bound: the integer ALU, three instructions a byte and round and about ten in the last walk; the
// bytes are read five times, from the last-level cache after the first. 134 MB in 0.36 ms where the
// host core took 110 ms.
//
// Version 2 of the snapshot format sums every 1 MiB block of the file from the offset basis: the BLOCKS forms walk
// all blocks of a piece at once, a block's runs as 64 workgroups of the same launches. Blocks begin and end anywhere in
// a run (the rows are aligned in device memory, not in the file): the bytes before a block's first whole run and
// behind its last are walked by one lane, fewer than 64 of each. Host threads, four blocks side by side each, took 0.9 ms
// for a block that is alone and 1.5 for 32. Host threads -> this, load / capture: 8 layers of 79 rows (1.3 MB) 1.00 /
// 0.97 -> 0.19 / 0.17 ms, 16 of 1,000 (33 MB) 3.05 / 3.7 -> 1.46 / 1.46.
#include "internal.h"

#include <algorithm>

namespace itak {

namespace {

constexpr uint64_t kPrime = 0x00000100000001b3ull;  // hash.rs:16
constexpr uint32_t kThreads = 256;
constexpr uint32_t kRun = kFnvRun;  // bytes a thread walks
static_assert(kRun == 64, "four 16-byte loads a thread");

// p^(kRun * 2^k)
struct Powers {
    uint64_t p[32];
};

__device__ __forceinline__ uint64_t power(const Powers &t, uint32_t e) {
    uint64_t r = 1;
#pragma unroll 1
    for (uint32_t k = 0; e; ++k, e >>= 1)
        if (e & 1) r *= t.p[k];
    return r;
}

// How a pair of bits is carried: bits 0..1 = the end for start 0, bits 2..3 = for start 1; the
// ends for 2 and 3 are those with the upper bit flipped.
constexpr uint32_t kIdentity = 0u | (1u << 2);
__device__ __forceinline__ uint32_t carry(uint32_t f, uint32_t v) { return ((f >> (2 * (v & 1))) & 3) ^ (v & 2); }
__device__ __forceinline__ uint32_t then(uint32_t first, uint32_t second) {
    return carry(second, first & 3) | (carry(second, first >> 2) << 2);
}

// Bytes [0, bytes) of a piece are bytes file_at .. of the file, and belong to its blocks first_block ..
struct FnvPiece {
    uint64_t file_at, bytes;
    uint32_t first_block, blocks;
};
constexpr uint32_t kBlockBits = 20;                                                // 1 MiB, kItkvSumBlock
constexpr uint32_t kBlockGroups = (1u << kBlockBits) / kRun / kThreads;            // workgroups a block
static_assert(kBlockGroups == 64, "a workgroup a lane");
// What the piece holds of a block: bytes [lo, head) before its first whole run, its runs, bytes [tail, hi) behind them.
struct FnvPart {
    uint64_t lo, head, tail, hi;
    uint32_t run0, runs;
    bool begins;  // else it goes on from the piece before, or from the file's header
    __device__ __forceinline__ FnvPart(const FnvPiece &p, uint32_t block) {
        const uint64_t from = uint64_t(p.first_block + block) << kBlockBits, to = from + (1ull << kBlockBits);
        begins = from >= p.file_at && from != 0;
        lo = from > p.file_at ? from - p.file_at : 0;
        hi = min(p.bytes, to - p.file_at);
        head = min((lo + kRun - 1) / kRun * kRun, hi);
        tail = max(head, hi / kRun * kRun);
        run0 = uint32_t(head / kRun);
        runs = uint32_t((tail - head) / kRun);
    }
};
__device__ __forceinline__ uint64_t walk_bytes(const unsigned char *bytes, uint64_t from, uint64_t to, uint64_t h) {
#pragma unroll 1
    for (uint64_t i = from; i < to; ++i) h = (h ^ bytes[i]) * kPrime;
    return h;
}
// The runs [run0, end) of a workgroup.
template <bool BLOCKS>
__device__ __forceinline__ void runs_of_group(const FnvPiece &piece, uint32_t runs, uint32_t &run0, uint32_t &end) {
    if constexpr (BLOCKS) {
        const FnvPart part(piece, blockIdx.x / kBlockGroups);
        const uint32_t at = min(blockIdx.x % kBlockGroups * kThreads, part.runs);
        run0 = part.run0 + at;
        end = run0 + min(kThreads, part.runs - at);
    } else {
        run0 = blockIdx.x * kThreads;
        end = min(runs, run0 + kThreads);
    }
}

// Carries of the lanes before this one (exclusive), and of the whole workgroup.
__device__ __forceinline__ uint32_t scan_carries(uint32_t f, uint32_t *lds, uint32_t *all) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = f;
#pragma unroll
    for (uint32_t s = 1; s < 64; s <<= 1) {
        const uint32_t before = __shfl_up(inc, s);
        if (lane >= s) inc = then(before, inc);
    }
    if (lane == 63) lds[wave] = inc;
    __syncthreads();
    uint32_t base = kIdentity, total = kIdentity;
#pragma unroll
    for (uint32_t w = 0; w < kThreads / 64; ++w) {
        if (w == wave) base = total;
        total = then(total, lds[w]);
    }
    const uint32_t before = __shfl_up(inc, 1);
    *all = total;
    return lane == 0 ? base : then(base, before);
}

__device__ __forceinline__ void load_run(const unsigned char *bytes, uint32_t run, uint32_t (&w)[kRun / 4]) {
    const uint4 *src = reinterpret_cast<const uint4 *>(bytes + uint64_t(run) * kRun);
#pragma unroll
    for (uint32_t i = 0; i < kRun / 16; ++i) {
        const uint4 v = src[i];
        w[4 * i] = v.x, w[4 * i + 1] = v.y, w[4 * i + 2] = v.z, w[4 * i + 3] = v.w;
    }
}

typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));

// The pair of bits this workgroup's runs start from: what the chain's start (`state`, bits 2*pair and up) becomes over
// the workgroups before it, whose carries the round left in `carries`. Every workgroup composes them for itself, 2,048 at
// most, where a launch of one workgroup stood between two rounds: six launches a piece instead of ten, captures of 1 and
// 2.6 MB 138 -> 128 and 186 -> 172 us.
template <bool BLOCKS>
__device__ __forceinline__ uint32_t start_pair(const uint8_t *carries, uint64_t state, uint32_t pair, uint32_t *lds) {
    const uint32_t first = BLOCKS ? blockIdx.x / kBlockGroups * kBlockGroups : 0, count = blockIdx.x - first;
    const uint32_t each = (count + kThreads - 1) / kThreads;
    uint32_t f = kIdentity, all;
    for (uint32_t i = threadIdx.x * each; i < min(count, (threadIdx.x + 1) * each); ++i) f = then(f, carries[first + i]);
    (void)scan_carries(f, lds, &all);
    return carry(all, uint32_t(state >> (2 * pair)) & 3);
}

// Round `pair`: bits 2*pair, 2*pair + 1 of the low byte. run_state[i]: the bits of run i's start
// known before this round, and above them (from bit 8) the carry from its workgroup's start that
// the last round left. Round 0 also starts the chains of the blocks that begin in the piece.
template <bool BLOCKS>
__global__ __launch_bounds__(kThreads) void fnv_round(const unsigned char *__restrict__ bytes, uint32_t runs, FnvPiece piece,
                                                      uint32_t pair, uint16_t *__restrict__ run_state,
                                                      const uint8_t *__restrict__ last_carry,
                                                      uint8_t *__restrict__ group_carry,
                                                      unsigned long long *__restrict__ state) {
    __shared__ uint32_t lds[kThreads / 64], lds_start[kThreads / 64];
    if constexpr (BLOCKS) {
        const uint32_t block = blockIdx.x / kBlockGroups;
        if (pair == 0 && blockIdx.x % kBlockGroups == 0 && threadIdx.x == 0) {
            const FnvPart part(piece, block);
            if (part.begins) state[piece.first_block + block] = walk_bytes(bytes, part.lo, part.head, 0xcbf29ce484222325ull);  // hash.rs:14
        }
        state += piece.first_block + block;
    }
    uint32_t run0, end;
    runs_of_group<BLOCKS>(piece, runs, run0, end);
    const uint32_t run = run0 + threadIdx.x;
    const uint32_t start = pair ? start_pair<BLOCKS>(last_carry, *state, pair - 1, lds_start) : 0;
    uint32_t f = kIdentity, known = 0;
    if (run < end) {
        uint32_t w[kRun / 4];
        load_run(bytes, run, w);
        if (pair) {
            const uint32_t s = run_state[run];
            known = (s & 0xff) | carry(s >> 8, start) << (2 * (pair - 1));
        }
        uint32_t x = known | ((known | (1u << (2 * pair))) << 16);
#pragma unroll
        for (uint32_t i = 0; i < kRun / 4; ++i)
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
                // byte b of the word in both halves, the other bytes zero
                x ^= __builtin_amdgcn_perm(w[i], w[i], 0x0c000c00u | (b << 16) | b);
                x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(ushort2v, x) * ushort2v{0xb3, 0xb3});
            }
        f = ((x >> (2 * pair)) & 3) | (((x >> (16 + 2 * pair)) & 3) << 2);
    }
    uint32_t all;
    const uint32_t before = scan_carries(f, lds, &all);
    if (run < end) run_state[run] = uint16_t(known | (before << 8));
    if (threadIdx.x == 0) group_carry[blockIdx.x] = uint8_t(all);
}

__device__ __forceinline__ uint64_t sum_workgroup(uint64_t v, uint64_t *lds) {
#pragma unroll
    for (uint32_t s = 32; s; s >>= 1) v += __shfl_down(v, s);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    return lds[0] + lds[1] + lds[2] + lds[3];
}

// Every run in 64 bits from its low byte, less what that byte contributes by itself, joined per
// workgroup as of the workgroup's last run.
template <bool BLOCKS>
__global__ __launch_bounds__(kThreads) void fnv_walk(const unsigned char *__restrict__ bytes, uint32_t runs, FnvPiece piece,
                                                     const uint16_t *__restrict__ run_state,
                                                     const uint8_t *__restrict__ last_carry,
                                                     const unsigned long long *__restrict__ state, Powers powers,
                                                     unsigned long long *__restrict__ group_sum) {
    __shared__ uint64_t lds[kThreads / 64];
    __shared__ uint32_t lds_start[kThreads / 64];
    const uint32_t start = start_pair<BLOCKS>(last_carry, state[BLOCKS ? piece.first_block + blockIdx.x / kBlockGroups : 0], 3,
                                              lds_start);
    uint32_t run0, end;
    runs_of_group<BLOCKS>(piece, runs, run0, end);
    const uint32_t run = run0 + threadIdx.x;
    uint64_t part = 0;
    if (run < end) {
        uint32_t w[kRun / 4];
        load_run(bytes, run, w);
        const uint32_t s = run_state[run];
        const uint64_t low = (s & 0xff) | (carry(s >> 8, start) << 6);
        uint64_t h = low;
#pragma unroll
        for (uint32_t i = 0; i < kRun / 4; ++i)
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) h = (h ^ ((w[i] >> (8 * b)) & 0xff)) * kPrime;
        part = (h - low * powers.p[0]) * power(powers, end - 1 - run);
    }
    const uint64_t sum = sum_workgroup(part, lds);
    if (threadIdx.x == 0) group_sum[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kThreads) void fnv_join(uint32_t runs, uint32_t groups, Powers powers,
                                                     const unsigned long long *__restrict__ group_sum,
                                                     unsigned long long *__restrict__ state) {
    __shared__ uint64_t lds[kThreads / 64];
    uint64_t part = 0;
    const uint32_t each = (groups + kThreads - 1) / kThreads;
    const uint32_t from = threadIdx.x * each, to = min(groups, from + each);
    for (uint32_t g = from; g < to; ++g)  // Horner: runs * 256 bytes from one group to the next
        part = part * (g + 1 == groups ? power(powers, runs - g * kThreads) : powers.p[8]) + group_sum[g];
    if (from < to) part *= power(powers, runs - min(runs, to * kThreads));
    const uint64_t sum = sum_workgroup(part, lds);
    if (threadIdx.x == 0) *state = *state * power(powers, runs) + sum;
}

// And of a piece's blocks, with the bytes behind their runs.
__global__ __launch_bounds__(kThreads) void fnv_join_blocks(const unsigned char *__restrict__ bytes, FnvPiece piece, Powers powers,
                                                            const unsigned long long *__restrict__ group_sum,
                                                            unsigned long long *__restrict__ state) {
    const uint32_t block = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (block >= piece.blocks) return;
    const FnvPart part(piece, block);
    const uint32_t upto = (lane + 1) * kThreads;
    uint64_t sum = group_sum[block * kBlockGroups + lane] * power(powers, part.runs - min(part.runs, upto));
#pragma unroll
    for (uint32_t s = 32; s; s >>= 1) sum += __shfl_down(sum, s);
    if (lane != 0) return;
    const uint64_t h = state[piece.first_block + block] * power(powers, part.runs) + sum;
    state[piece.first_block + block] = walk_bytes(bytes, part.tail, part.hi, h);
}

const Powers &powers_of_run() {
    static const Powers powers = [] {
        Powers t;
        uint64_t p = 1;
        for (uint32_t i = 0; i < kRun; ++i) p *= kPrime;
        for (uint64_t &x : t.p) {
            x = p;
            p *= p;
        }
        return t;
    }();
    return powers;
}

}  // namespace

uint64_t fnv_scratch_bytes(uint64_t bytes) {
    const uint64_t runs = bytes / kRun, blocks = (bytes >> kBlockBits) + 2;
    const uint64_t groups = std::max((runs + kThreads - 1) / kThreads, blocks * kBlockGroups);
    return 256 + (groups * 8 + groups * 2 + runs * 2 + 1023) / 256 * 256;
}

template <bool BLOCKS>
static void launch_rounds(const unsigned char *bytes, uint32_t runs, const FnvPiece &piece, uint32_t groups, void *scratch,
                          unsigned long long *state, hipStream_t stream) {
    unsigned long long *group_sum = static_cast<unsigned long long *>(scratch);
    uint16_t *run_state = reinterpret_cast<uint16_t *>(group_sum + groups);
    uint8_t *carries[2] = {reinterpret_cast<uint8_t *>(run_state + runs), reinterpret_cast<uint8_t *>(run_state + runs) + groups};
    for (uint32_t pair = 0; pair < 4; ++pair)
        launch_kernel(fnv_round<BLOCKS>, groups, kThreads, 0, stream, bytes, runs, piece, pair, run_state, carries[~pair & 1],
                      carries[pair & 1], state);
    launch_kernel(fnv_walk<BLOCKS>, groups, kThreads, 0, stream, bytes, runs, piece, run_state, carries[1], state, powers_of_run(),
                  group_sum);
}

hipError_t launch_fnv(const void *data, uint64_t bytes, void *scratch, unsigned long long *state, hipStream_t stream) {
    const uint32_t runs = uint32_t(bytes / kRun), groups = (runs + kThreads - 1) / kThreads;
    if (runs == 0) return hipSuccess;
    launch_rounds<false>(static_cast<const unsigned char *>(data), runs, FnvPiece{}, groups, scratch, state, stream);
    launch_kernel(fnv_join, 1, kThreads, 0, stream, runs, groups, powers_of_run(), static_cast<unsigned long long *>(scratch), state);
    return hipGetLastError();
}

hipError_t launch_fnv_blocks(const void *data, uint64_t bytes, uint64_t file_at, void *scratch, unsigned long long *states,
                             hipStream_t stream) {
    if (bytes == 0) return hipSuccess;
    const uint32_t first = uint32_t(file_at >> kBlockBits);
    const FnvPiece piece{file_at, bytes, first, uint32_t((file_at + bytes - 1) >> kBlockBits) - first + 1};
    const unsigned char *b = static_cast<const unsigned char *>(data);
    launch_rounds<true>(b, uint32_t(bytes / kRun), piece, piece.blocks * kBlockGroups, scratch, states, stream);
    launch_kernel(fnv_join_blocks, (piece.blocks + kThreads / 64 - 1) / (kThreads / 64), kThreads, 0, stream, b, piece,
                  powers_of_run(), static_cast<unsigned long long *>(scratch), states);
    return hipGetLastError();
}

}  // namespace itak
