// Host side of the C ABI: the pool, its slots, the per-slot bookkeeping that mirrors
// attention::KvCache (crates/attention/src/cache.rs) and cpu_compute::CpuCompute
// (crates/cpu-compute/src/cpu.rs), and the launch logic for the kernels in this directory.
// All validation happens here, in the reference's order, before anything is enqueued.
#include "../../include/itak_hip_kv.h"
#include "internal.h"
#include "host_ring.h"
#include "host_turns.h"
#include "load_room.h"
#include "itkv.h"

#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <ctime>
#include <string>
#include <vector>

using namespace itak;

// Split workspace of itak_attention_step_device_noalloc: see the notes at g_scratch_of_device.
// Host code never passes this name to a kernel or a memory call: it is a host-side handle,
// the device address comes from hipGetSymbolAddress.
static __device__ __align__(256) unsigned char scratch[16ull << 20];

namespace {

// One windowed layer's rows set aside by a checkpoint whose round is longer than the ring's
// headroom (the saved slots of cache.rs:678-697): `rows` positions from the layer's base on.
struct RingSave {
    uint32_t layer = 0;      // pool layer
    uint32_t rows = 0;
    uint64_t saved_off = 0;  // elements into the slot's side buffer
    uint64_t high0 = 0;      // the layer's high-water mark when the checkpoint was taken
};

struct LiveCheckpoint {
    bool live = false;
    uint64_t serial = 0;
    uint64_t max_round_tokens = 0;
    std::vector<uint64_t> bases;
    std::vector<RingSave> ring_saves;  // empty when the headroom covers the round
};

struct Slot {
    bool in_use = false;
    bool built = false;  // CpuCompute's KvState exists (cpu.rs:560-564)
    uint64_t cache_id = 0;
    uint64_t next_serial = 0;
    std::vector<uint64_t> appended;  // per layer: positions appended == next position
    // Per layer: one past the highest position ever written into the storage since it was
    // last fresh. Positions in [appended, high) were dropped by a rewind; on a windowed layer
    // their rows still sit in the ring and alias the positions one ring length below them.
    std::vector<uint64_t> high;
    // Per layer: the oldest position the storage was ever given. 0 for a sequence appended
    // from its start; the first restored position of a windowed layer filled from a snapshot,
    // which carries only the last `window` rows: nothing below it can come back into view.
    std::vector<uint64_t> floor;
    LiveCheckpoint cp;
};

// One layer of the pattern (attention::LayerKind, cache.rs:36-48) and where it lives.
struct LayerInfo {
    bool windowed = false;
    uint32_t index = 0;   // among the layers of its kind, which are stored together
    uint64_t window = 0;  // attention window; 0 on a global layer
    uint32_t ring = 0;    // storage rows of the ring (a multiple of 32); 0 on a global layer
};

struct ErrorState {
    std::string message;
    itak_error_info info{};
};

thread_local ErrorState g_create_error;

// ---- the split workspace of the allocation-free entry point --------------------------------
// itak_attention_step_device_noalloc may not allocate, so its split workspace is this array:
// every device the library runs on holds a copy until the process ends. The first part holds
// exchange words for launches that merge their own splits (all empty between launches, like
// the pool's own exchange buffer); the rest takes the partials of launches that leave the
// merge to a second launch. In host code the array's name is only a handle: the address the
// kernels get is looked up once per device (bind_scratch) and kept here.
constexpr uint64_t kScratchBytes = sizeof(scratch);
constexpr uint64_t kScratchExchangeBytes = 8ull << 20;
constexpr int kMaxDevices = 64;
unsigned char *g_scratch_of_device[kMaxDevices];
std::mutex g_scratch_mutex;
// Every pool and stream of a device shares the device's copy of the array. Eager calls are kept
// apart by an event (made with the address, at set-up): recorded behind every allocation-free
// step on the stream it ran on, and waited for, on the device, by the next such step when that
// one runs on another stream. Calls made while their stream is being captured into a graph are
// outside this guard: nothing runs at the call, and when the replays run is the caller's matter.
struct ScratchGuard {
    hipEvent_t done = nullptr;     // behind the last eager allocation-free step of the device
    hipStream_t stream = nullptr;  // the stream that step ran on
    bool recorded = false;
};
ScratchGuard g_scratch_guard[kMaxDevices];
std::atomic<uint64_t> g_next_cache_id{1};  // cache.rs:32

}  // namespace

// rope_base^(-2i/rotary_dim), i < rotary_dim/2, computed on the host and kept on the device, table after
// table behind the pool's planes (or in an allocation of their own).
struct RopeFreqTable {
    float base;
    uint32_t rotary;
    bool made;                   // by an eager launch: whatever runs later finds it
    unsigned long long capture;  // the capture that holds a launch that makes it, and on which stream
    hipStream_t stream;
};

// One item's query rows against its slot; fills the split plan.
struct PlanInput {
    uint32_t slot;
    uint32_t rows;
    uint32_t pos0;
    uint32_t kv_len;
    uint32_t kv_lo;  // oldest position the item's queries may see
};

struct itak_pool {
    itak_pool_config cfg{};
    std::vector<RopeFreqTable> rope_tables;
    double *rope_dev = nullptr;      // room for rope_tables_max tables of head_dim / 2
    bool rope_apart = false;         // in an allocation of their own
    uint32_t rope_tables_max = 0;
    // Global layers and windowed layers are two groups of planes with their own row capacity:
    // `g` (capacity_rows per plane) and `gw` (the longest ring per plane). Within a group the
    // layers are consecutive, so the kernels that walk several layers take (group base,
    // group geometry, index within the group).
    PoolGeom g{};
    PoolGeom gw{};
    std::vector<LayerInfo> layers;
    uint32_t global_layers = 0, windowed_layers = 0;
    // Rows a windowed layer's ring holds beyond its window: the longest block one step may
    // append there and the deepest rewind (crates/wgpu-compute/src/session.rs:235-249,
    // 5376-5428 give the algebra).
    uint64_t headroom = 0;
    int elem_f16 = 0;
    uint32_t elem_bytes = 4;
    uint64_t row = 0;         // kv_heads * head_dim
    uint64_t rows_limit = 0;  // positions a slot may hold on a global layer (the configured capacity)
    unsigned char *base = nullptr;    // global layers
    unsigned char *base_w = nullptr;  // windowed layers (inside the same allocation)
    uint64_t bytes = 0;
    hipStream_t stream = nullptr;
    std::vector<Slot> slots;
    // Device scratch, grown on demand and reused: staging for host-pointer calls and
    // split partials.
    unsigned char *stage = nullptr;
    uint64_t stage_bytes = 0;
    float *ws = nullptr;
    uint64_t ws_floats = 0;
    float *prep = nullptr;  // prepared Q and K rows of a prep step
    uint64_t prep_floats = 0;
    // Exchange buffer of split-K launches that merge their splits themselves: 64-bit words,
    // every one holding the empty pattern whenever no such launch is running; word 0 counts
    // the consumers that gave up waiting (checked by itak_pool_synchronize).
    unsigned long long *xws = nullptr;
    uint64_t xws_words = 0;
    uint32_t spin_limit = 1u << 17;  // looks at the buffer a consumer makes before it gives up
    // This device's copy of the static split workspace, and whether the call in progress must
    // use it instead of the pool's own buffers (itak_attention_step_device_noalloc).
    unsigned char *scratch_dev = nullptr;
    bool no_alloc_call = false;
    bool scratch_exchange_used = false;  // its give-up counter is then looked at too
    bool merge_in_launch = false;
    // ITAK_POOL_DIE_MERGE: split-K launches whose units deal out evenly over the compute dies
    // merge each unit's splits on its die (attn_splitk_f16_die.hip): one ticket word per unit, then the count of
    // workgroups that found themselves on another die than planned.
    bool die_merge = false;
    uint32_t *die_words = nullptr;
    bool q_two_halves = false;  // ITAK_POOL_Q_TWO_HALVES
    bool prep_by_launch = false;  // ITAK_POOL_PREP_BY_LAUNCH
    // Per slot: the side buffer of a deep checkpoint's ring rows, kept for the next one
    // (cache.rs:620-625: allocated once per cache, not once per round).
    std::vector<void *> ring_saved;
    std::vector<uint64_t> ring_saved_bytes;
    // Pinned host memory for the host-pointer attention call: its small inputs are packed here
    // and go up in one copy; its kernels write the output here directly.
    unsigned char *hstage = nullptr;
    unsigned char *hstage_dev = nullptr;  // the device's address of it
    uint64_t hstage_half = 0;             // bytes of each of its two halves (host_turns.h)
    HostTurns turns;
    // Pinned slots through which snapshot rows move between ordinary host memory and the device.
    HostRing ring;
    // Plan of the step in progress, and the slots it has named (by the number of the step).
    std::vector<PlanInput> plan, active;
    AttnBatch block_plan;  // the block kernel's plan of the step at hand, where its price was asked (KernelChoice)
    std::vector<uint64_t> named;
    uint64_t step_number = 0;
    uint32_t call_number = 0;  // what the last host-pointer call asked to be told when done
    mutable ErrorState err;
};

namespace {

// ------------------------------------------------------------------------------ debug channel
// attention::diag (crates/attention/src/diag.rs:13-33,71-79): off by default; the switch or
// ITAK_HIP_KV_DEBUG in the environment (any value but "0" or empty, looked up at every event as
// the reference looks its variable up) turns one stderr line per event on.
std::atomic<bool> g_debug_enabled{false};

bool diag_enabled() {
    if (g_debug_enabled.load(std::memory_order_relaxed)) return true;
    const char *v = getenv("ITAK_HIP_KV_DEBUG");
    return v && v[0] != '\0' && !(v[0] == '0' && v[1] == '\0');
}

__attribute__((format(printf, 1, 2))) void diag_emit(const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    fprintf(stderr, "[itak_hip_kv::diag] %s\n", buf);
}

#define ITAK_DIAG(...)                          \
    do {                                        \
        if (diag_enabled()) diag_emit(__VA_ARGS__); \
    } while (0)

// ------------------------------------------------------------------------------ errors

itak_status set_error(ErrorState &e, int32_t code, const char *what, uint64_t a, uint64_t b,
                      uint64_t c, uint64_t d, const char *fmt, ...) {
    e.info = itak_error_info{};
    e.info.code = code;
    if (what) snprintf(e.info.what, sizeof(e.info.what), "%s", what);
    e.info.a = a;
    e.info.b = b;
    e.info.c = c;
    e.info.d = d;
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    e.message = buf;
    ITAK_DIAG("refused code=%d: %s", int(code), buf);  // every refusal says why
    return code;
}

#define ULL(x) static_cast<unsigned long long>(x)

// The Display texts of AttentionError (crates/attention/src/error.rs:129-214).
itak_status zero_dimension(ErrorState &e, const char *what) {
    return set_error(e, ITAK_ZERO_DIMENSION, what, 0, 0, 0, 0, "%s must be positive, got 0", what);
}
itak_status invalid_window(ErrorState &e, uint64_t window) {
    return set_error(e, ITAK_INVALID_WINDOW, nullptr, window, 0, 0, 0,
                     "sliding window must be positive, got %llu", ULL(window));
}
itak_status size_overflow(ErrorState &e, const char *what) {
    return set_error(e, ITAK_SIZE_OVERFLOW, what, 0, 0, 0, 0, "%s: element count overflows usize",
                     what);
}
itak_status shape_mismatch(ErrorState &e, const char *what, uint64_t expected, uint64_t actual) {
    return set_error(e, ITAK_SHAPE_MISMATCH, what, expected, actual, 0, 0,
                     "%s: got %llu, expected %llu", what, ULL(actual), ULL(expected));
}
itak_status invalid_layer(ErrorState &e, uint64_t layer, uint64_t layer_count) {
    return set_error(e, ITAK_INVALID_LAYER, nullptr, layer, layer_count, 0, 0,
                     "layer %llu out of range, cache has %llu layers", ULL(layer),
                     ULL(layer_count));
}
itak_status out_of_order(ErrorState &e, uint64_t layer, uint64_t expected, uint64_t actual) {
    return set_error(e, ITAK_OUT_OF_ORDER_POSITION, nullptr, layer, expected, actual, 0,
                     "layer %llu appends must be in order: expected position %llu, got %llu",
                     ULL(layer), ULL(expected), ULL(actual));
}
itak_status non_divisible(ErrorState &e, uint64_t q_heads, uint64_t kv_heads) {
    return set_error(e, ITAK_NON_DIVISIBLE_HEADS, nullptr, q_heads, kv_heads, 0, 0,
                     "%llu query heads do not divide evenly across %llu KV heads", ULL(q_heads),
                     ULL(kv_heads));
}
itak_status no_visible_keys(ErrorState &e, uint64_t position) {
    return set_error(e, ITAK_NO_VISIBLE_KEYS, nullptr, position, 0, 0, 0,
                     "query at position %llu has no visible keys", ULL(position));
}
itak_status checkpoint_busy(ErrorState &e) {
    return set_error(e, ITAK_CHECKPOINT_BUSY, nullptr, 0, 0, 0, 0,
                     "a checkpoint is already outstanding on this cache; release it before "
                     "taking another");
}
itak_status stale_checkpoint(ErrorState &e, uint64_t serial) {
    return set_error(e, ITAK_STALE_CHECKPOINT, nullptr, serial, 0, 0, 0,
                     "checkpoint %llu is not this cache's live checkpoint (already released or "
                     "foreign)",
                     ULL(serial));
}
itak_status range_exceeded(ErrorState &e, uint64_t layer, uint64_t position, uint64_t limit) {
    return set_error(e, ITAK_CHECKPOINT_RANGE_EXCEEDED, nullptr, layer, position, limit, 0,
                     "layer %llu append at position %llu is outside the live checkpoint's saved "
                     "range (first unsaved position %llu); refusing so a later rewind cannot meet "
                     "a slot it cannot restore",
                     ULL(layer), ULL(position), ULL(limit));
}
itak_status not_fresh(ErrorState &e, uint64_t layer, uint64_t appended) {
    return set_error(e, ITAK_BULK_RESTORE_NOT_FRESH, nullptr, layer, appended, 0, 0,
                     "layer %llu already holds %llu appended positions; bulk restore installs "
                     "into a fresh layer only",
                     ULL(layer), ULL(appended));
}
itak_status rewind_range(ErrorState &e, uint64_t layer, uint64_t base, uint64_t appended,
                         uint64_t target) {
    return set_error(e, ITAK_REWIND_OUT_OF_RANGE, nullptr, layer, base, appended, target,
                     "rewind target %llu is outside layer %llu's checkpoint range [%llu, %llu]",
                     ULL(target), ULL(layer), ULL(base), ULL(appended));
}
itak_status hip_error(ErrorState &e, hipError_t code, const char *doing) {
    return set_error(e, ITAK_HIP_ERROR, doing, uint64_t(code), 0, 0, 0, "%s: HIP error %d (%s)",
                     doing, int(code), hipGetErrorString(code));
}
itak_status invalid_argument(ErrorState &e, const char *what) {
    return set_error(e, ITAK_INVALID_ARGUMENT, what, 0, 0, 0, 0, "invalid argument: %s", what);
}
itak_status capacity_exceeded(ErrorState &e, uint64_t layer, uint64_t need, uint64_t capacity) {
    return set_error(e, ITAK_CAPACITY_EXCEEDED, nullptr, layer, need, capacity, 0,
                     "layer %llu would hold %llu positions but the pool's slots hold %llu",
                     ULL(layer), ULL(need), ULL(capacity));
}
itak_status unsupported(ErrorState &e, const char *what) {
    return set_error(e, ITAK_UNSUPPORTED, what, 0, 0, 0, 0, "unsupported: %s", what);
}

#define HIP_TRY(pool, call, doing)                                   \
    do {                                                             \
        hipError_t _e = (call);                                      \
        if (_e != hipSuccess) return hip_error((pool)->err, _e, doing); \
    } while (0)

// ------------------------------------------------------------------------------ helpers

Slot *find_slot(itak_pool *pool, uint32_t slot) {
    if (slot >= pool->slots.size() || !pool->slots[slot].in_use) return nullptr;
    return &pool->slots[slot];
}

const PoolGeom &geom_of(const itak_pool *pool, uint64_t layer) {
    return pool->layers[layer].windowed ? pool->gw : pool->g;
}

void *layer_base(itak_pool *pool, uint64_t layer) {
    const LayerInfo &L = pool->layers[layer];
    return (L.windowed ? pool->base_w : pool->base) +
           L.index * geom_of(pool, layer).layer_stride * pool->elem_bytes;
}

// Positions stored and visible (cache.rs:154-159) and the oldest of them (cache.rs:162-164).
uint64_t stored_of(const itak_pool *pool, const Slot &s, uint64_t layer) {
    const LayerInfo &L = pool->layers[layer];
    return L.windowed ? std::min(s.appended[layer], L.window) : s.appended[layer];
}
uint64_t first_visible(const itak_pool *pool, const Slot &s, uint64_t layer) {
    return s.appended[layer] - stored_of(pool, s, layer);
}

void advance(Slot &s, uint64_t layer, uint64_t rows) {
    s.appended[layer] += rows;
    s.high[layer] = std::max(s.high[layer], s.appended[layer]);
}

itak_status ensure_stage(itak_pool *pool, uint64_t bytes) {
    if (bytes <= pool->stage_bytes) return ITAK_OK;
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing staging");
    if (pool->stage) HIP_TRY(pool, hipFree(pool->stage), "free staging");
    pool->stage = nullptr;
    pool->stage_bytes = 0;
    uint64_t want = std::max<uint64_t>(bytes + bytes / 2, 1u << 20);
    HIP_TRY(pool, hipMalloc(reinterpret_cast<void **>(&pool->stage), want), "allocate staging");
    pool->stage_bytes = want;
    return ITAK_OK;
}

// The rotation frequencies of (base, rotary_dim) in device memory: the same expression, in the same f64
// libm, as rope.rs:99-116 and rope_interleaved.rs:103-114 evaluate on the host. Made on first use by a
// launch that carries them as its argument, ahead of the step on its stream: nothing is allocated and
// nothing waits (as an allocation and a copy of its own it made a preparing decode step's first call
// 31.6 us instead of 22.6; taking the powers in the kernel 19.5). A first use inside a capture is captured
// with the step, whose replays then make the table themselves, always the same; for everything outside
// that graph it has yet to be made. Null when there is no room for another table: the preparation kernel
// then takes the powers itself.
const double *rope_freq_table(itak_pool *pool, float base, uint32_t rotary) {
    if (!(base > 1.0f) || rotary < 2) return nullptr;
    size_t at = 0;
    while (at < pool->rope_tables.size() && !(pool->rope_tables[at].base == base && pool->rope_tables[at].rotary == rotary)) ++at;
    double *dev = pool->rope_dev + at * (pool->g.head_dim / 2);
    if (at < pool->rope_tables.size() && pool->rope_tables[at].made) return dev;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long capture = 0;
    bool known = hipStreamGetCaptureInfo(pool->stream, &status, &capture) == hipSuccess;
    if (!known) (void)hipGetLastError();
    const bool captured = known && status == hipStreamCaptureStatusActive;
    if (at == pool->rope_tables.size()) {
        if (at == pool->rope_tables_max) return nullptr;
        pool->rope_tables.push_back(RopeFreqTable{base, rotary, false, 0, nullptr});
    }
    RopeFreqTable &table = pool->rope_tables[at];
    if (captured && table.capture == capture && table.stream == pool->stream) return dev;
    for (uint32_t first = 0; first < rotary / 2; first += kFillDoubles) {
        FillDoubles a;
        a.n = std::min<uint32_t>(kFillDoubles, rotary / 2 - first);
        for (uint32_t i = 0; i < a.n; ++i)
            a.v[i] = std::pow(double(base), -double(2 * (first + i)) / double(rotary));
        if (launch_fill_doubles(dev + first, a, pool->stream) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
    }
    table.made = known && status == hipStreamCaptureStatusNone;
    table.capture = captured ? capture : 0;
    table.stream = pool->stream;
    return dev;
}

itak_status ensure_workspace(itak_pool *pool, uint64_t floats) {
    if (floats > pool->ws_floats) {
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing workspace");
        if (pool->ws) HIP_TRY(pool, hipFree(pool->ws), "free workspace");
        pool->ws = nullptr;
        pool->ws_floats = 0;
        uint64_t want = std::max<uint64_t>(floats + floats / 2, 1u << 18);
        HIP_TRY(pool, hipMalloc(reinterpret_cast<void **>(&pool->ws), want * sizeof(float)),
                "allocate split workspace");
        pool->ws_floats = want;
    }
    return ITAK_OK;
}

// (Re)fills the exchange buffer with the empty pattern and zeroes its give-up counter.
itak_status clean_exchange(itak_pool *pool) {
    HIP_TRY(pool, launch_fill_words(pool->xws, pool->xws_words, kExchangeEmptyWord, pool->stream),
            "fill the split exchange buffer");
    HIP_TRY(pool, launch_fill_words(pool->xws, 1, 0, pool->stream), "zero the give-up counter");
    return ITAK_OK;
}

itak_status ensure_exchange(itak_pool *pool, uint64_t words) {
    if (words > pool->xws_words) {
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing the exchange buffer");
        if (pool->xws) HIP_TRY(pool, hipFree(pool->xws), "free the exchange buffer");
        pool->xws = nullptr;
        pool->xws_words = 0;
        const uint64_t want = std::max<uint64_t>(words + words / 2, 1u << 17);
        HIP_TRY(pool, hipMalloc(reinterpret_cast<void **>(&pool->xws), want * 8),
                "allocate the split exchange buffer");
        pool->xws_words = want;
        return clean_exchange(pool);
    }
    return ITAK_OK;
}

itak_status ensure_prep(itak_pool *pool, uint64_t floats) {
    if (floats > pool->prep_floats) {
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing prep scratch");
        if (pool->prep) HIP_TRY(pool, hipFree(pool->prep), "free prep scratch");
        pool->prep = nullptr;
        pool->prep_floats = 0;
        uint64_t want = std::max<uint64_t>(floats + floats / 2, 1u << 16);
        HIP_TRY(pool, hipMalloc(reinterpret_cast<void **>(&pool->prep), want * sizeof(float)),
                "allocate prep scratch");
        pool->prep_floats = want;
    }
    return ITAK_OK;
}

uint64_t align_up(uint64_t x, uint64_t a) { return (x + a - 1) / a * a; }

constexpr uint64_t kHostWord = 256;  // bytes at the head of the pinned staging kept for the completion word
constexpr uint64_t kHostHalf = 1u << 19;  // smallest half of the rest
// Making and freeing pinned memory takes some 45 us, as much as a small call, which a program with a pool
// for every sequence would pay for each. A pool that closes leaves a staging of the smallest size for the
// next one: at most one a device (a megabyte), kept until the process ends.
std::atomic<unsigned char *> g_spare_hstage[kMaxDevices];
itak_status ensure_hstage(itak_pool *pool, uint64_t half_bytes) {
    if (half_bytes <= pool->hstage_half) return ITAK_OK;
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing pinned staging");
    pool->turns.drained();
    if (pool->hstage) HIP_TRY(pool, hipHostFree(pool->hstage), "free pinned staging");
    pool->hstage = nullptr;
    pool->hstage_half = 0;
    const uint64_t half = align_up(std::max<uint64_t>(half_bytes + half_bytes / 2, kHostHalf), 256);
    if (half == kHostHalf) pool->hstage = g_spare_hstage[pool->cfg.device].exchange(nullptr);
    if (!pool->hstage)
        HIP_TRY(pool, hipHostMalloc(reinterpret_cast<void **>(&pool->hstage), kHostWord + 2 * half, hipHostMallocDefault),
                "allocate pinned staging");
    memset(pool->hstage, 0, kHostWord);  // the completion word of a call must not start out matching
    void *mapped = nullptr;
    HIP_TRY(pool, hipHostGetDevicePointer(&mapped, pool->hstage, 0), "map pinned staging");
    pool->hstage_dev = static_cast<unsigned char *>(mapped);
    pool->hstage_half = half;
    return ITAK_OK;
}

hipStream_t stream_of(const HostTurns &turns) { return static_cast<hipStream_t>(const_cast<void *>(turns.stream())); }

// Waits until nothing of earlier host-pointer calls runs, on whichever stream they ran.
itak_status drain_host_calls(itak_pool *pool) {
    if (hipStreamSynchronize(stream_of(pool->turns)) != hipSuccess) {
        (void)hipGetLastError();  // (the caller has destroyed that stream)
        HIP_TRY(pool, hipDeviceSynchronize(), "wait for an earlier call's launches");
    }
    pool->turns.drained();
    return ITAK_OK;
}

// The staging of a pool that closes; nothing else uses it once the host-pointer calls' launches have ended.
void release_hstage(itak_pool *pool) {
    const bool quiet = !pool->turns.running() || drain_host_calls(pool) == ITAK_OK;
    unsigned char *none = nullptr;
    if (pool->hstage && !(quiet && pool->hstage_half == kHostHalf &&
                          g_spare_hstage[pool->cfg.device].compare_exchange_strong(none, pool->hstage)))
        (void)hipHostFree(pool->hstage);
    pool->hstage = nullptr;
    pool->hstage_half = 0;
}

// ---- host-pointer attention calls ------------------------------------------------------
// Such a call is dominated by its trips over the host link and by its launches, not by its
// kernels. Its inputs are packed into pinned memory and read from there by the device, its output
// is written into pinned memory by whichever kernel makes it, and the host watches for it there:
// finding out from the runtime that a stream has drained costs several microseconds more.
// Calls that move more than kHostPacked copy their arrays as they lie.
constexpr uint64_t kHostPacked = 4ull << 20;
// Up to here the host watches the output itself: every word of it is set beforehand to a pattern
// that no arithmetic makes, and the output is there when the pattern is gone. (A NaN that came in
// with a caller's row could carry it: such a call ends on the runtime's word.) Larger outputs are
// announced by a one-thread launch; 2.4 us of host time and a launch behind the merge.
constexpr uint64_t kHostWatched = 64ull << 10;
constexpr uint32_t kNotYet = 0xffffa5c3u;
// Inputs up to this size go up by a launch that reads them over the link (a copy-engine command
// costs 7 us at 20 KB, the launch 3); above it the copy engine's rate wins.
constexpr uint64_t kHostByLaunch = 256ull << 10;

struct HostCall {
    unsigned char *in = nullptr;       // where the host packs the inputs
    unsigned char *in_dev = nullptr;   // the same memory as the device sees it
    float *out_dev = nullptr;          // the output's place as the device sees it
    uint64_t out_at = 0;               // and its offset in the pinned staging
    uint64_t out_count = 0;            // floats
};

itak_status begin_host_call(itak_pool *pool, uint64_t in_bytes, uint64_t out_count, HostCall &c) {
    // Layout: [completion word, 256 bytes] [inputs, output] [inputs, output], the halves in turn. The
    // word sits at a fixed place, so it only ever holds call numbers, which only grow.
    const uint64_t in_room = align_up(in_bytes, 256);
    itak_status st = ITAK_OK;
    if (pool->turns.must_drain(pool->stream)) st = drain_host_calls(pool);
    if (st == ITAK_OK) st = ensure_hstage(pool, in_room + out_count * 4);
    if (st != ITAK_OK) return st;
    const uint64_t at = kHostWord + pool->turns.begin(pool->stream) * pool->hstage_half;
    c.in = pool->hstage + at;
    c.in_dev = pool->hstage_dev + at;
    c.out_at = at + in_room;
    c.out_dev = reinterpret_cast<float *>(pool->hstage_dev + c.out_at);
    c.out_count = out_count;
    if (out_count * 4 <= kHostWatched)
        std::fill_n(reinterpret_cast<uint32_t *>(pool->hstage + c.out_at), out_count, kNotYet);
    return ITAK_OK;
}

// Everything of the call is on the stream: its output to `out`.
itak_status finish_host_call(itak_pool *pool, const HostCall &c, float *out) {
    const bool watched = c.out_count * 4 <= kHostWatched;
    const uint32_t number = ++pool->call_number ? pool->call_number : ++pool->call_number;
    if (!watched)
        HIP_TRY(pool, launch_signal_done(reinterpret_cast<uint32_t *>(pool->hstage_dev), number, pool->stream),
                "launch completion signal");
    const unsigned char *from = pool->hstage + c.out_at;
    unsigned char *to = reinterpret_cast<unsigned char *>(out);
    const uint64_t bytes = c.out_count * 4;
    timespec t0{};
    clock_gettime(CLOCK_MONOTONIC, &t0);
    // The host looks for 0.3 ms before it asks the runtime (which also reports a failed launch, and
    // is what a call that takes longer falls back to).
    auto look_until = [&](auto ready) {
        for (uint32_t spin = 0;; ++spin) {
            if (ready()) return true;
            __builtin_ia32_pause();
            if ((spin & 63u) != 63u) continue;
            timespec t1{};
            clock_gettime(CLOCK_MONOTONIC, &t1);
            if ((t1.tv_sec - t0.tv_sec) * 1000000000ll + (t1.tv_nsec - t0.tv_nsec) > 300000) return false;
        }
    };
    if (!watched) {
        const volatile uint32_t *seen = reinterpret_cast<const volatile uint32_t *>(pool->hstage);
        if (!look_until([&] { return __atomic_load_n(seen, __ATOMIC_ACQUIRE) == number; }))
            HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after attention");
        pool->turns.drained();
        memcpy(out, from, bytes);
        return ITAK_OK;
    }
    // A piece is copied first and looked at in the copy, so that what was looked at is what the
    // caller gets.
    for (uint64_t at = 0; at < bytes;) {
        const uint64_t n = std::min<uint64_t>(512, bytes - at);
        const bool arrived = look_until([&] {
            asm volatile("" ::: "memory");
            memcpy(to + at, from + at, n);
            const uint32_t *w = reinterpret_cast<const uint32_t *>(to + at);
            uint32_t missing = 0;
            for (uint64_t i = 0; i < n / 4; ++i) missing |= w[i] == kNotYet;
            return missing == 0;
        });
        if (!arrived) {
            HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after attention");
            pool->turns.drained();
            memcpy(out, from, bytes);
            return ITAK_OK;
        }
        at += n;
    }
    pool->turns.seen();
    return ITAK_OK;
}

// The address of this device's copy of `scratch`, looked up on first use with the device
// current; the exchange part is filled with the empty pattern then (a kernel on the null
// stream, waited for). Later calls return the kept address.
hipError_t bind_scratch(int device, unsigned char **out) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_of_device[device]) {
        unsigned char *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!ptr) return hipErrorInvalidSymbol;
        e = launch_fill_words(reinterpret_cast<unsigned long long *>(ptr), kScratchExchangeBytes / 8,
                              kExchangeEmptyWord, nullptr);
        if (e == hipSuccess) e = launch_fill_words(reinterpret_cast<unsigned long long *>(ptr), 1, 0, nullptr);
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (e != hipSuccess) return e;
        e = hipEventCreateWithFlags(&g_scratch_guard[device].done, hipEventDisableTiming);
        if (e != hipSuccess) return e;
        g_scratch_of_device[device] = ptr;
    }
    *out = g_scratch_of_device[device];
    return hipSuccess;
}

// Before an allocation-free step is enqueued on `stream`: if the device's last such step ran on
// another stream, this one waits for it on the device. Returns whether the stream is being
// captured (the guard then stands aside).
hipError_t scratch_guard_enter(int device, hipStream_t stream, bool *capturing) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(stream, &status);
    if (e != hipSuccess) return e;
    *capturing = status != hipStreamCaptureStatusNone;
    if (*capturing) return hipSuccess;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ScratchGuard &g = g_scratch_guard[device];
    if (g.recorded && g.stream != stream) return hipStreamWaitEvent(stream, g.done, 0);
    return hipSuccess;
}
// After it: the event now stands behind this step.
hipError_t scratch_guard_leave(int device, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ScratchGuard &g = g_scratch_guard[device];
    const hipError_t e = hipEventRecord(g.done, stream);
    if (e == hipSuccess) {
        g.stream = stream;
        g.recorded = true;
    }
    return e;
}

// What the launches of one attention call need beyond their inputs and outputs.
struct WorkspaceNeed {
    uint64_t partial_floats = 0;   // split partials for a merge launch
    uint64_t exchange_words = 0;   // exchange words of launches that merge their own splits
};

// Builds the work list and launches the attention kernels. q/out are device pointers.
// f16 pools at head_dim 128 with up to 64 query vectors per KV head (decode and
// speculative blocks) take the MFMA split-K kernel; everything else the generic kernel.
// Either way a second small launch merges the split partials.
// True when a batch takes the MFMA split-K kernel (which can also fuse the append).
bool takes_splitk_f16(const itak_pool *pool, const PlanInput *in, uint32_t n, uint64_t q_heads,
                      const uint32_t *q_pos_dev) {
    const uint32_t group = uint32_t(q_heads / pool->g.kv_heads);
    uint32_t max_rows = 0;
    for (uint32_t i = 0; i < n; ++i) max_rows = std::max(max_rows, in[i].rows);
    // Decode and speculative blocks (up to 64 query vectors per KV head, up to 8 new rows):
    // the split-K kernel, which also appends the new rows. Its 64-vector variant and the
    // block kernel (wavefronts split the query vectors, K/V shared through LDS) attend at the
    // same speed on a 7-row block; the fused append decides (one launch less per layer).
    constexpr uint32_t max_vec = 64;
    return pool->elem_f16 && q_pos_dev == nullptr && max_rows * group <= max_vec &&
           attn_splitk_f16_supports(pool->g, group, max_rows);  // g and gw differ in capacity only
}

// The f32-arithmetic matrix kernel takes what has no kernel of its own: f16 pools at other head dims
// or with groups above 16, f32 pools at other head dims. Its 16-byte loads and stores ask for
// tensors aligned to that (every row is a multiple of 16 bytes when head_dim is one of four
// floats); others, odd head dims and explicit positions run on the general kernel.
// It also takes f16 steps of up to 16 query vectors per KV head at head dims 64, 96 and 256, where
// the block kernel has nothing to share between its wavefronts: no LDS ring to fill before the first
// product, runs down to one block per wavefront, short contexts left whole. 32 Q / 4 KV heads, us a
// layer, block kernel -> this: one slot at 1,500 rows 9.5 -> 8.9, 11.3 -> 8.9, 15.8 -> 12.7 (head_dim
// 64, 96, 256), 4 slots at 300 10.2 -> 7.2, 11.7 -> 8.1, 14.9 -> 13.3. At 256 a wavefront's operands
// leave room for one workgroup per compute unit, so that launches of more than one block per wavefront
// of the device and less than two run two rounds of blocks for little more than one round's work: those
// stay with the block kernel (8 slots of 2,000 rows 21.8 against 23.5; of 3,000 rows 34.3 -> 28.5).
bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
bool takes_splitk_any(const itak_pool *pool, const PlanInput *in, uint32_t n, uint64_t q_heads, const float *q_dev,
                      const float *out_dev, const uint32_t *q_pos_dev) {
    const uint32_t group = uint32_t(q_heads / pool->g.kv_heads);
    uint32_t max_rows = 0;
    uint64_t blocks = 0;
    for (uint32_t i = 0; i < n; ++i) {
        max_rows = std::max(max_rows, in[i].rows);
        blocks += uint64_t(pool->g.kv_heads) * ((in[i].kv_len + 31) / 32 - in[i].kv_lo / 32);
    }
    const uint64_t round = 4 * uint64_t(compute_units());
    const bool has_own = !pool->elem_f16 ? attn_splitk_f32_supports(pool->g, group, max_rows)
                                         : attn_prefill_f16_supports(pool->g, group) &&
                                               (pool->g.head_dim == 128 || max_rows * group > 16 ||
                                                (pool->g.head_dim == 256 && blocks > round && blocks <= 2 * round));
    return q_pos_dev == nullptr && aligned16(q_dev) && aligned16(out_dev) &&
           !takes_splitk_f16(pool, in, n, q_heads, q_pos_dev) && !has_own &&
           attn_splitk_any_supports(pool->g, group, max_rows);
}

// Whether a call's output lies over its queries, or over new rows that its launch brings along. Steps by channels
// (attn_whole_f16.hip, attn_parts_halves.hip) have several workgroups read what one of them writes over, whichever comes
// first; the other forms read all of a (slot, KV head)'s inputs in the workgroup that writes its output, or a launch before the
// merge that does. (The gate is read by the thread that writes over it.)
bool shares_memory(const itak_pool *pool, const PlanInput *in, uint32_t n, uint64_t q_heads, const float *out_dev,
                   const float *q_dev, const float *k_new, const float *v_new) {
    uint64_t rows = 0;
    for (uint32_t i = 0; i < n; ++i) rows += in[i].rows;
    const uint64_t q_bytes = rows * q_heads * pool->g.head_dim * sizeof(float), kv_bytes = rows * pool->row * sizeof(float);
    auto over = [&](const float *p, uint64_t bytes) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p), o = reinterpret_cast<uintptr_t>(out_dev);
        return p && a < o + q_bytes && o < a + bytes;
    };
    return over(q_dev, q_bytes) || over(k_new, kv_bytes) || over(v_new, kv_bytes);
}

// Clears a batch's plan and names its items' places; q rows counted from q_row0. Returns their rows.
uint32_t start_batch(AttnBatch &b, const PlanInput *in, uint32_t count, uint32_t q_row0) {
    b.n = count;  // (cleared item by item: all 64 are three kilobytes)
    b.total_blocks = b.rows_per_block = b.tiles = b.fold_units = b.whole_on_eight = b.parts = b.scale_scores = b.tiled = b.on_eight = b.half_blocks = 0;
    b.two_halves = b.tile_sets = b.tile_waves = b.tile_exact = 0;
    b.plan_cost = 0.0f;
    b.partial_limit = 0;
    uint32_t rows = 0;
    for (uint32_t i = 0; i < count; ++i) {
        AttnItem &it = b.item[i];
        it = AttnItem{};
        it.slot = in[i].slot;
        it.rows = in[i].rows;
        it.pos0 = in[i].pos0;
        it.q_row0 = q_row0 + rows;
        it.kv_len = in[i].kv_len;
        it.kv_lo = in[i].kv_lo;
        rows += in[i].rows;
    }
    return rows;
}

// Steps on f16 pools at head_dim 128 that the tiles kernel (attn_tiles_f16.hip) takes from the split-K kernel
// and the block kernel, and in which form.
//
// Against the block kernel the two planners' costs decide; `kBlockLaunch` and `kBlockAppends` put that
// kernel's walk and merge on the tiles' scale (medians over the shapes the tiles' figures were fitted on). The pick is
// 1.4 % behind the better of the two kernels there, before the margins below, and in two of 549 shapes slower than the block
// kernel by more than 2 %. 32 Q / 4 KV heads, us a layer, block kernel -> tiles: 61 rows on 0 / 300 / 1,000 12.4 / 17.9 /
// 19.1 -> 7.5 / 8.9 / 12.3, on a window of 2,048 18.8 -> 15.9; 24 rows on 4,099 18.4 -> 14.1; 128 rows on 1,000
// 24.5 -> 13.8; 512 rows on 0 20.1 -> 17.1. The block kernel keeps many rows on long contexts (192 rows on 12,000:
// 62.5 against 73.3). The fit has no launches of several slots of which one brings 128 rows and more: there the
// tiles take 3 to 8 us beyond their estimate, and `kLongBesideOthers` is added. Over 320 random steps of 1 to 42 slots, most
// of them decode rows and short blocks beside a chunk, on which the estimates without it chose the tiles, these took 0.74 of
// the block kernel's time and 14 steps more than 2 % longer (17 slots of seven rows beside 244 22.6 -> 27.4); with it 0.75,
// and two, 8 % at most (320 others: one, 4 %). 3 / 31 / 7 decode rows at 500 / 1,500 / 2,000 beside 128 / 128 / 64 rows on 1,000 / 0 /
// 2,000: 22.0 / 40.1 / 21.8 -> 14.2 / 31.7 / 16.7.
//
// Estimates within 8 % of each other are the block kernel's (`kAhead`): near ties on contexts beyond the fit were not
// ties (71 rows on 18,376 44.0 -> 51.5, 248 on 8,241 at 8 KV heads 55.6 -> 64.4). Over 1,255 random steps, 617 with the keys
// out of the caches, the tiles took 0.749 of the block kernel's time without the margin, 15 more than 2 % longer and 17 % at
// worst; with it 0.754, six and 6 %.
//
// Against the split-K kernel, whose 16-vector steps are the better ones throughout (the rows come in through
// LDS, the loads stream): steps of more vectors while the keys are at most one and a half blocks per compute
// unit and the launch is its longest chain (7 rows at 300 9.7 -> 8.3, at 1,000 9.6 -> 8.6, 8 slots at 300 10.4 -> 9.7).
// Beyond, each tile's pass over the keys shows (keys that are not in the last-level cache: 4 slots of four rows at 8,192
// 20.4 against 21.7). Several slots: contexts that kernel leaves whole, and as whole tiles, so up to 16 blocks, 8 from
// eight KV heads on, where it has twice the workgroups; one slot also split, from 17 blocks on. With the keys out of the
// caches, split-K -> tiles, 400 positions (13 blocks): 4 KV heads 1 / 3 slots of eight rows 8.8 / 9.7 -> 8.4 / 9.3, 8 KV
// heads 2 of six 9.2 -> 10.0; a window of 512 (17 blocks): 1 slot of eight rows 9.5 -> 9.0 split (10.6 whole), 2 / 5 of
// three 9.9 / 10.6 -> 10.8 / 11.5 split (11.4 / 11.8 whole). 160 random steps there 6 % faster on average, 7 % slower at worst,
// 120 with the keys in the caches 7 and 6 %. Softcaps
// outside [2, 1024] stay there too: the tiles round the queries with 2 log2(e) / softcap on, the split-K kernel caps the
// scores, and beyond those the factor takes queries out of f16's range, or into its subnormals, that are inside it there.
struct KernelChoice {
    bool in_place = false;         // out shares memory with what the launch reads (`shares_memory`)
    TilesPlan tiles;               // sets = 0: another kernel
    bool block = false;            // pool->block_plan is the block kernel's plan of the step,
    bool block_appends = false;    // in a launch that brings the rows along or not,
    uint32_t block_partials = 0;   // and its partials
};
KernelChoice choose_tiles(itak_pool *pool, uint64_t layer, const PlanInput *in, uint32_t n, uint64_t q_heads, float softcap,
                          bool prepares, bool brings_rows, bool no_alloc) {
    KernelChoice choice;
    const uint32_t group = uint32_t(q_heads / pool->g.kv_heads);
    uint32_t max_rows = 0;
    uint64_t blocks = 0;
    uint32_t most = 0;
    for (uint32_t i = 0; i < n; ++i) {
        max_rows = std::max(max_rows, in[i].rows);
        const uint32_t held = (in[i].kv_len + 31) / 32 - in[i].kv_lo / 32;
        most = std::max(most, held);
        blocks += uint64_t(pool->g.kv_heads) * held;
    }
    if (!pool->elem_f16 || pool->q_two_halves || n == 0 || n > uint32_t(kMaxBatchItems) ||
        !attn_tiles_f16_supports(pool->g, group, max_rows))
        return choice;
    const bool splitk = takes_splitk_f16(pool, in, n, q_heads, nullptr);
    if (splitk && (prepares || pool->merge_in_launch || pool->die_merge || max_rows * group <= 16 ||
                   (softcap > 0.0f && (softcap < 2.0f || softcap > 1024.0f)) ||
                   (most > (pool->g.kv_heads >= 8 ? 8u : 16u) && (n > 1 || most <= 16)) ||
                   2 * blocks > 3 * uint64_t(compute_units())))
        return choice;
    const PoolGeom &geom = geom_of(pool, layer);
    const uint32_t window = uint32_t(std::min<uint64_t>(pool->layers[layer].window, 0xffffffffu));
    const uint64_t limit = no_alloc ? kScratchBytes - kScratchExchangeBytes : 0;
    AttnBatch &b = pool->block_plan;
    start_batch(b, in, n, 0);
    float below = INFINITY;
    if (!splitk) {
        constexpr float kBlockLaunch = 6.8f, kBlockAppends = 6.4f, kLongBesideOthers = 5.0f, kAhead = 0.92f;
        uint32_t most_blocks = 0;
        for (uint32_t i = 0; i < n; ++i) most_blocks = std::max(most_blocks, item_block_count(b.item[i]));
        const bool appends = brings_rows && attn_prefill_f16_appends(pool->g, group, max_rows, most_blocks);
        choice.block_partials = attn_prefill_f16_plan(geom, b, group, uint32_t(q_heads), window, appends);
        choice.block = true;
        choice.block_appends = appends;
        below = kAhead * (b.plan_cost + kBlockLaunch + (brings_rows && !appends ? kBlockAppends : 0.0f)) -
                (n > 1 && max_rows >= 128 ? kLongBesideOthers : 0.0f);
    }
    attn_tiles_f16_choose(geom, b, uint32_t(q_heads), window, brings_rows, splitk, limit, below, choice.tiles);
    if (no_alloc && choice.tiles.sets) {
        // (The allocation-free call refuses a step by the same plans as without the tiles, see run_attention.)
        AttnBatch m;
        start_batch(m, in, n, 0);
        const uint64_t partials = splitk ? attn_splitk_f16_plan(geom, m, uint32_t(q_heads), false, true)
                                         : attn_prefill_f16_plan(geom, m, group, uint32_t(q_heads), window, false);
        if (partials * (pool->g.head_dim + 2) * sizeof(float) > limit) choice.tiles = TilesPlan{};
    }
    return choice;
}

// k_new / v_new non-null = the rows are not in the cache yet and the kernel appends them
// (only valid when takes_splitk_f16 holds).
itak_status run_attention(itak_pool *pool, uint64_t layer, const PlanInput *in, uint32_t n,
                          const float *q_dev, float *out_dev, const uint32_t *q_pos_dev,
                          uint64_t q_heads, float scale, float softcap,
                          const float *k_new = nullptr, const float *v_new = nullptr,
                          const FoldedParams *folded = nullptr, WorkspaceNeed *need_only = nullptr,
                          const KernelChoice *chosen = nullptr) {
    const uint32_t group = uint32_t(q_heads / pool->g.kv_heads);
    uint32_t max_rows = 0;
    for (uint32_t i = 0; i < n; ++i) max_rows = std::max(max_rows, in[i].rows);
    // (A step has asked already, since who appends hangs on it.)
    const KernelChoice choice = chosen ? *chosen
                                : q_pos_dev ? KernelChoice{}
                                            : choose_tiles(pool, layer, in, n, q_heads, softcap, folded && folded->prep_on,
                                                           false, need_only || pool->no_alloc_call);
    const bool in_place = chosen ? choice.in_place : shares_memory(pool, in, n, q_heads, out_dev, q_dev, k_new, v_new);
    const TilesPlan &form = choice.tiles;
    const bool tiles = form.sets != 0;
    const bool mfma = !tiles && takes_splitk_f16(pool, in, n, q_heads, q_pos_dev);
    // Blocks of many rows (prefill chunks) on the same pools take the MFMA prefill kernel.
    const bool any = takes_splitk_any(pool, in, n, q_heads, q_dev, out_dev, q_pos_dev);
    const bool prefill = !tiles && !mfma && !any && pool->elem_f16 && q_pos_dev == nullptr &&
                         attn_prefill_f16_supports(pool->g, group);
    // Decode steps and short blocks on f32 pools of head_dim 128: the f32 MFMA split-K kernel.
    const bool f32fast = !pool->elem_f16 && q_pos_dev == nullptr &&
                         attn_splitk_f32_supports(pool->g, group, max_rows);
    const uint32_t rpb =
        (tiles || mfma || prefill || f32fast || any) ? 0 : attn_generic_rows_per_block(group, pool->g.head_dim);
    if (!tiles && !mfma && !prefill && !f32fast && !any && rpb == 0)
        return unsupported(pool->err, "head_dim above 256 or GQA group too wide");
    const uint32_t tile = attn_generic_tile(pool->g.head_dim);
    constexpr uint64_t kTargetBlocks = 1024;  // about four workgroups per CU
    const LayerInfo &L = pool->layers[layer];
    const PoolGeom &geom = geom_of(pool, layer);
    const uint32_t window = uint32_t(std::min<uint64_t>(L.window, 0xffffffffu));

    uint32_t q_row0 = 0;
    for (uint32_t first = 0; first < n; first += kMaxBatchItems) {
        const uint32_t count = std::min<uint32_t>(kMaxBatchItems, n - first);
        // (Planned already where the choice has asked for the block kernel's price; such steps are one batch.)
        const bool planned = prefill && choice.block && !need_only && !pool->no_alloc_call &&
                             choice.block_appends == (k_new != nullptr);
        AttnBatch own;
        AttnBatch &b = planned ? pool->block_plan : own;
        uint32_t total_rows = 0;
        if (planned)
            for (uint32_t i = 0; i < count; ++i) total_rows += in[i].rows;
        else
            total_rows = start_batch(b, in + first, count, q_row0);
        q_row0 += total_rows;
        b.two_halves = prefill && pool->q_two_halves && pool->g.head_dim == 128 ? 1 : 0;
        // (At head_dim 128 a step is refused when the best plan of a launch without its rows outgrows the static
        // workspace; a launch that brings them along is cut otherwise, up to twice the partials, and takes the
        // best plan that fits, as every launch at the other head dims does.)
        b.partial_limit = (need_only || pool->no_alloc_call) && (pool->g.head_dim != 128 || k_new)
                              ? kScratchBytes - kScratchExchangeBytes : 0;
        uint32_t partials = 0;
        if (planned) {
            partials = choice.block_partials;
        } else if (tiles) {
            partials = attn_tiles_f16_plan(geom, b, uint32_t(q_heads), form);
        } else if (mfma) {
            partials = attn_splitk_f16_plan(geom, b, uint32_t(q_heads), folded && folded->prep_on,
                                            !pool->q_two_halves && !pool->merge_in_launch,
                                            !pool->q_two_halves && !pool->merge_in_launch && !pool->die_merge && !in_place);
        } else if (prefill) {
            partials = attn_prefill_f16_plan(geom, b, group, uint32_t(q_heads), window, k_new != nullptr);
        } else if (f32fast || any) {
            partials = attn_splitk_f32_plan(geom, pool->elem_f16, b, uint32_t(q_heads),
                                            any && max_rows * group <= 16 ? attn_splitk_any_groups_per_cu(geom) : 2,
                                            need_only || pool->no_alloc_call ? kScratchBytes - kScratchExchangeBytes : 0,
                                            !in_place);
        } else {
            b.rows_per_block = rpb;
            uint64_t key_work = 0;
            for (uint32_t i = 0; i < count; ++i) {
                const uint64_t qblocks = (b.item[i].rows + rpb - 1) / rpb;
                key_work += qblocks * pool->g.kv_heads * (b.item[i].kv_len - b.item[i].kv_lo);
            }
            const uint64_t kps = align_up(
                std::max<uint64_t>((key_work + kTargetBlocks - 1) / kTargetBlocks, tile), tile);
            uint32_t block0 = 0;
            for (uint32_t i = 0; i < count; ++i) {
                AttnItem &it = b.item[i];
                const uint32_t keys = it.kv_len - it.kv_lo;
                it.keys_per_split = uint32_t(kps);
                it.splits = uint32_t((keys + kps - 1) / kps);
                if (it.splits == 0) it.splits = 1;
                if (it.splits > 1024) {  // the merge kernel holds at most 1024 weights
                    it.keys_per_split = uint32_t(align_up((keys + 1023) / 1024, tile));
                    it.splits = (keys + it.keys_per_split - 1) / it.keys_per_split;
                }
                const uint32_t qblocks = (it.rows + rpb - 1) / rpb;
                it.block0 = block0;
                it.ws0 = partials;
                block0 += qblocks * pool->g.kv_heads * it.splits;
                if (it.splits > 1) partials += it.rows * uint32_t(q_heads) * it.splits;
            }
            b.total_blocks = block0;
        }
        // Split-K launches merge their splits themselves where the plan allows it (the gate,
        // when there is one, must then be applied by that kernel: its preparing variants).
        const float *gate = folded ? folded->gate : nullptr;
        const bool prepares = folded && folded->prep_on && mfma;
        uint64_t exchange_words = 0;
        if (mfma && pool->merge_in_launch && (!gate || prepares))
            exchange_words = attn_splitk_f16_plan_exchange(geom, b, uint32_t(q_heads));
        // Or on the units' compute dies, when the batch deals out evenly over them and is not
        // one the single-row decode kernel takes.
        AttnBatch bd;
        DieMap dm;
        uint32_t die_partials = 0;
        if (mfma && pool->die_merge && !exchange_words && !pool->q_two_halves) {
            bd = AttnBatch{};
            dm = DieMap{};
            AttnParams probe{};
            probe.g = geom;
            probe.group = group;
            if (prepares || !attn_decode_f16_takes(probe, b))
                die_partials = attn_splitk_f16_plan_die(geom, b, uint32_t(q_heads), bd, dm);
        }
        const bool on_die = die_partials != 0;
        if (on_die) partials = die_partials;
        const AttnBatch &bl = on_die ? bd : b;  // the batch the attention launch takes
        const uint64_t partial_floats = uint64_t(partials) * (pool->g.head_dim + 2);
        if (need_only) {  // planning only: nothing is allocated, launched or changed
            need_only->exchange_words = std::max(need_only->exchange_words, exchange_words);
            if (!exchange_words)
                need_only->partial_floats = std::max(need_only->partial_floats, partial_floats);
            continue;
        }
        float *ws = nullptr;
        if (pool->no_alloc_call) {
            // The caller has checked the need against the static workspace's two parts.
            ws = reinterpret_cast<float *>(exchange_words ? pool->scratch_dev
                                                          : pool->scratch_dev + kScratchExchangeBytes);
        } else {
            // (A chunk's windowed and global layers are split differently; the first one's partials leave
            // room for the others': growing costs a wait and an allocation, 600 us in the middle of a forward.)
            const uint64_t floats = tiles && !form.exact && partials ? std::max<uint64_t>(partial_floats, 1u << 21) : partial_floats;
            itak_status st = exchange_words ? ensure_exchange(pool, exchange_words) : ensure_workspace(pool, floats);
            if (st != ITAK_OK) return st;
            ws = exchange_words ? reinterpret_cast<float *>(pool->xws) : pool->ws;
        }
        // The reference's line (attention.rs:147-155) plus which kernel takes the launch, and in the forms that the
        // planners of some choose between, its wavefronts a workgroup.
        if (diag_enabled()) {
            // (Steps by channels run on eight, in that many parts of the channels, or of that many channel tiles each.)
            char by_channels[24];
            snprintf(by_channels, sizeof by_channels, mfma ? "8,parts=%u" : "8,tiles=%u", b.parts);
            const char *waves = b.parts ? by_channels : tiles ? (b.tile_waves == 8 ? "8" : "4")
                                : !f32fast && !any ? "-" : b.half_blocks ? "4,half_blocks" : b.on_eight ? "8" : "4";
            const char *kernel = tiles ? "tiles_f16" : mfma ? (b.parts ? "whole_f16" : "splitk_f16") : prefill ? "prefill_f16"
                                 : f32fast ? "splitk_f32" : any ? (b.parts ? "parts_halves" : "splitk_any") : "generic";
            uint32_t splits = 0;
            uint64_t view_len = 0;
            for (uint32_t i = 0; i < count; ++i) {
                splits = std::max(splits, bl.item[i].splits);
                view_len = std::max<uint64_t>(view_len, b.item[i].kv_len - b.item[i].kv_lo);
            }
            diag_emit("gqa_attention layer=%llu items=%u queries=%u q_heads=%llu kv_heads=%llu "
                      "view_len=%llu window=%u scale=%g softcap=%g kernel=%s workgroups=%u splits=%u "
                      "wavefronts=%s fused_append=%d merge=%s",
                      ULL(layer), count, total_rows, ULL(q_heads), ULL(pool->g.kv_heads), ULL(view_len),
                      window, double(scale), double(softcap),
                      kernel, bl.total_blocks, splits, waves, int(k_new != nullptr && (tiles || mfma || f32fast || any || prefill)),
                      partials == 0 ? "none" : on_die ? "on_die" : exchange_words ? "in_launch" : "launch");
        }
        AttnParams p{};
        p.layer_base = layer_base(pool, layer);
        p.g = geom;
        p.window = window;
        p.ring_blocks = L.ring / kVBlock;
        p.q = q_dev;
        p.out = out_dev;
        p.q_pos = q_pos_dev;
        p.ws = ws;
        p.exchange = exchange_words ? 1 : 0;
        p.fold_units = prefill ? b.fold_units : 0;
        {
            uint64_t rows_read = 0;
            for (uint32_t i = 0; i < count; ++i) rows_read += b.item[i].kv_len - b.item[i].kv_lo;
            const uint64_t layer_bytes = rows_read * 2 * pool->g.kv_heads * pool->g.head_dim *
                                         (pool->elem_f16 ? 2 : 4);
            p.kv_streams = layer_bytes * pool->layers.size() > (uint64_t(512) << 20) ? 1 : 0;  // twice the cache: well clear of it
        }
        p.spin_limit = pool->spin_limit;
        p.scale_scores = b.scale_scores;
        p.k_new = (tiles || mfma || f32fast || any || prefill) ? k_new : nullptr;  // the caller passes them only to
        p.v_new = (tiles || mfma || f32fast || any || prefill) ? v_new : nullptr;  // launches that append themselves
        p.q_heads = uint32_t(q_heads);
        p.group = group;
        p.group_magic = (65536u + group - 1) / group;
        p.scale = scale;
        p.softcap = softcap;
        // The gate is applied by whoever writes the output: the merge for items of several
        // splits; for items of one split the split-K kernel, which only its preparing
        // variants can; otherwise a launch of its own over the chunk's rows.
        bool merged_only = mfma || prefill;
        for (uint32_t i = 0; i < count; ++i) merged_only = merged_only && bl.item[i].splits > 1;
        const bool gate_folded = gate && (prepares || tiles || (mfma && merged_only));
        if (on_die) {
            dm.tickets = pool->die_words;
            dm.faults = pool->die_words + kDieTicketBytes / sizeof(uint32_t);
            dm.gate = gate_folded ? gate : nullptr;
            HIP_TRY(pool,
                    launch_attn_splitk_f16_die(p, bd, dm, partials, pool->stream,
                                               prepares ? folded : nullptr),
                    "launch split-K attention");
        } else if (mfma) {
            HIP_TRY(pool,
                    launch_attn_splitk_f16(p, b, partials, max_rows, pool->stream,
                                           prepares ? folded : nullptr, pool->q_two_halves),
                    "launch split-K attention");
        } else if (tiles) {
            HIP_TRY(pool, launch_attn_tiles_f16(p, b, partials, gate, pool->stream), "launch tiles of attention");
        } else if (prefill) {
            HIP_TRY(pool, launch_attn_prefill_f16(p, b, partials, pool->stream),
                    "launch block attention");
        } else if (f32fast) {
            HIP_TRY(pool, launch_attn_splitk_f32(p, b, partials, pool->stream),
                    "launch f32 split-K attention");
        } else if (any) {
            HIP_TRY(pool, launch_attn_splitk_any(pool->elem_f16, p, b, partials, pool->stream),
                    "launch split-K attention of any head_dim");
        } else {
            HIP_TRY(pool, launch_attn_generic(pool->elem_f16, p, b, partials, pool->stream),
                    "launch attention");
        }
        if (!exchange_words && !on_die)
            HIP_TRY(pool, launch_attn_combine(p, b, partials, total_rows, (tiles || mfma || prefill || f32fast || any) ? 1 : 0,
                                              pool->stream, gate_folded ? gate : nullptr),
                    "launch split merge");
        if (gate && !gate_folded) {
            const uint64_t q_width = q_heads * pool->g.head_dim;
            const uint64_t at = uint64_t(q_row0 - total_rows) * q_width;
            HIP_TRY(pool, launch_attn_gate(out_dev + at, gate + at, total_rows * q_width, pool->stream),
                    "launch attention gate");
        }
    }
    return ITAK_OK;
}

float default_scale(uint64_t head_dim) {  // attention.rs:35-37
    return 1.0f / std::sqrt(static_cast<float>(head_dim));
}

// Appends `rows` rows per item from device sources; the caller has validated everything.
itak_status run_append(itak_pool *pool, uint64_t layer, const itak_batch_item *items, uint32_t n,
                       const float *k_dev, const float *v_dev) {
    const LayerInfo &L = pool->layers[layer];
    const PoolGeom &geom = geom_of(pool, layer);
    // A long run of one slot's rows into blocked planes (a prefill chunk) moves by blocks. (At the head
    // dims that can attend; a block's rows of wider heads outgrow the LDS a launch may ask for.)
    constexpr uint32_t kChunkRows = 64;
    if (n == 1 && pool->elem_f16 && geom.v_block != 0 && geom.head_dim <= 256 && items[0].rows >= kChunkRows && aligned16(k_dev) && aligned16(v_dev) &&
        (!L.windowed || (L.ring % kVBlock == 0 && items[0].rows <= L.ring))) {
        const uint32_t slot = items[0].slot, rows = items[0].rows;
        HIP_TRY(pool, launch_append_chunk(layer_base(pool, layer), geom, slot, uint32_t(pool->slots[slot].appended[layer]), rows,
                                          L.windowed ? uint32_t(L.ring) : 0, k_dev, v_dev, pool->stream),
                "launch chunk append");
        advance(pool->slots[slot], layer, rows);
        return ITAK_OK;
    }
    uint32_t src_row = 0;
    for (uint32_t first = 0; first < n; first += kMaxBatchItems) {
        const uint32_t count = std::min<uint32_t>(kMaxBatchItems, n - first);
        AppendBatch b{};
        b.n = count;
        b.ring = L.ring;
        const uint32_t chunk_row0 = src_row;
        for (uint32_t i = 0; i < count; ++i) {
            const itak_batch_item &bi = items[first + i];
            b.item[i].slot = bi.slot;
            b.item[i].rows = bi.rows;
            b.item[i].pos0 = uint32_t(pool->slots[bi.slot].appended[layer]);
            b.item[i].src_row0 = src_row - chunk_row0;
            src_row += bi.rows;
        }
        b.total_rows = src_row - chunk_row0;
        HIP_TRY(pool,
                launch_append(layer_base(pool, layer), pool->elem_f16, geom, b,
                              k_dev + uint64_t(chunk_row0) * pool->row,
                              v_dev + uint64_t(chunk_row0) * pool->row, pool->stream),
                "launch append");
    }
    for (uint32_t i = 0; i < n; ++i) {
        advance(pool->slots[items[i].slot], layer, items[i].rows);
        ITAK_DIAG("append layer=%llu slot=%u rows=%u kind=%s stored=%llu", ULL(layer), items[i].slot,
                  items[i].rows, L.windowed ? "windowed" : "global",
                  ULL(pool->slots[items[i].slot].appended[layer]));
    }
    return ITAK_OK;
}

// The append preconditions of KvCache::append (cache.rs:445-471) for `rows` consecutive
// positions starting at the layer's next one; returns how many rows may be appended
// before a refusal (rows if none) and leaves that refusal in the error state.
// Positions a slot may hold on a layer: the configured capacity on a global layer; a ring
// never fills, its positions only have to stay well inside 32 bits.
uint64_t position_limit(const itak_pool *pool, uint64_t layer) {
    return pool->layers[layer].windowed ? 0xfff00000ull : pool->rows_limit;
}

itak_status check_append_rows(itak_pool *pool, Slot &s, uint64_t layer, uint64_t rows,
                              uint64_t *ok_rows) {
    uint64_t ok = rows;
    itak_status st = ITAK_OK;
    const uint64_t start = s.appended[layer];
    if (s.cp.live) {
        const uint64_t limit = s.cp.bases[layer] + s.cp.max_round_tokens;
        if (start + rows > limit) {
            ok = limit > start ? limit - start : 0;
            st = range_exceeded(pool->err, layer, start + ok, limit);
        }
    }
    const uint64_t rows_limit = position_limit(pool, layer);
    if (start + ok > rows_limit) {
        ok = rows_limit > start ? rows_limit - start : 0;
        st = capacity_exceeded(pool->err, layer, start + ok + 1, rows_limit);
    }
    *ok_rows = ok;
    return st;
}

// A block of a device step lands in a windowed layer's ring before its queries run, so it
// may be at most as long as the ring's headroom over the window.
itak_status check_block_rows(itak_pool *pool, uint64_t layer, uint64_t rows) {
    const LayerInfo &L = pool->layers[layer];
    if (!L.windowed || rows <= L.ring - L.window) return ITAK_OK;
    return set_error(pool->err, ITAK_CAPACITY_EXCEEDED, nullptr, layer, rows, L.ring - L.window, 0,
                     "a block of %llu rows does not fit the %llu rows of ring headroom of windowed "
                     "layer %llu; split the block or build the pool with a larger ring_headroom",
                     ULL(rows), ULL(L.ring - L.window), ULL(layer));
}

// Zero fill of rows [row_from, row_to) of every global layer of the listed slots.
itak_status scrub_rows(itak_pool *pool, const ZeroBatch &zb) {
    HIP_TRY(pool,
            launch_zero_rows(pool->base, pool->elem_f16, pool->g, 0, pool->global_layers, zb,
                             pool->stream),
            "launch row scrub");
    return ITAK_OK;
}

// Pointer kinds for restore sources. For memory the device can read in place, `usable`
// is the address a kernel should dereference.
enum class PtrKind { Device, PinnedHost, PlainHost };
PtrKind classify(const void *p, const void **usable) {
    *usable = p;
    hipPointerAttribute_t attr{};
    hipError_t e = hipPointerGetAttributes(&attr, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // an unknown pointer is ordinary host memory, not a failure
        return PtrKind::PlainHost;
    }
    if (attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged)
        return PtrKind::Device;
    if (attr.type == hipMemoryTypeHost) {
        if (attr.devicePointer) *usable = attr.devicePointer;
        return PtrKind::PinnedHost;
    }
    return PtrKind::PlainHost;
}

// The same for the many sources of one restore: a snapshot's layers usually lie in one or two
// device allocations, and the runtime's lookup costs microseconds a pointer (two lookups a
// layer and side were more host time than the gather of a 48-layer prefix takes the device).
// The extent of the last device allocation seen answers for every pointer inside it.
struct PtrClassifier {
    uintptr_t lo = 0, hi = 0;  // a device allocation already looked up
    PtrKind operator()(const void *p, const void **usable) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p);
        if (a >= lo && a < hi) {
            *usable = p;
            return PtrKind::Device;
        }
        const PtrKind kind = classify(p, usable);
        if (kind == PtrKind::Device) {
            hipDeviceptr_t base = nullptr;
            size_t size = 0;
            if (hipMemGetAddressRange(&base, &size, const_cast<void *>(p)) == hipSuccess && size) {
                lo = reinterpret_cast<uintptr_t>(base);
                hi = lo + size;
            } else {
                (void)hipGetLastError();
            }
        }
        return kind;
    }
};

// Rows the gather kernel cannot read where they lie: ordinary host memory, or a source that
// is not aligned to its element size (the payload of an encoded snapshot starts wherever
// its fingerprint ends).
bool must_stage(PtrClassifier &kind_of, const void *p, uint64_t elem_bytes) {
    const void *usable;
    return kind_of(p, &usable) == PtrKind::PlainHost ||
           reinterpret_cast<uintptr_t>(p) % elem_bytes != 0;
}

itak_status set_itkv_error(ErrorState &e, const ItkvError &err) {
    return set_error(e, err.code, "snapshot", err.a, err.b, 0, 0, "%s", err.message.c_str());
}

ItkvHeader to_internal(const itak_itkv_header &h) {
    ItkvHeader r;
    r.token_count = h.token_count;
    r.num_kv_heads = h.num_kv_heads;
    r.head_dim = h.head_dim;
    r.layer_count = h.layer_count;
    r.fingerprint_len = h.fingerprint_len;
    return r;
}
std::vector<ItkvLayer> to_internal(const itak_itkv_layer *layers, uint64_t n) {
    std::vector<ItkvLayer> r(n);
    for (uint64_t i = 0; i < n; ++i) {
        r[i].kind = layers[i].kind;
        r[i].window = layers[i].window;
        r[i].first_position = layers[i].first_position;
        r[i].rows = layers[i].rows;
    }
    return r;
}

}  // namespace

// ======================================================================== public ABI

namespace itak {

int32_t restore_decoded_itkv(itak_pool *pool, uint32_t slot, const uint8_t *b8, const ItkvHeader &h,
                             const std::vector<ItkvLayer> &ls, const char *expected_fingerprint,
                             uint64_t expected_fingerprint_len, const uint8_t *rows) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!find_slot(pool, slot)) return invalid_argument(pool->err, "slot is not in use");
    // restore_checked (snapshot.rs:351-371): geometry first, then the fingerprint.
    bool same = h.layer_count == pool->cfg.layer_count && h.num_kv_heads == pool->g.kv_heads &&
                h.head_dim == pool->g.head_dim;
    for (size_t i = 0; same && i < ls.size(); ++i)
        same = pool->layers[i].windowed
                   ? (ls[i].kind == ITAK_LAYER_WINDOWED && ls[i].window == pool->layers[i].window)
                   : ls[i].kind == ITAK_LAYER_GLOBAL;
    if (!same)
        return set_error(pool->err, ITAK_KV_GEOMETRY_MISMATCH, "snapshot", 0, 0, 0, 0,
                         "geometry mismatch: snapshot geometry (%llu layers, %llu KV heads, head "
                         "dim %llu) differs from the required geometry (%llu layers, %llu KV "
                         "heads, head dim %llu)",
                         ULL(h.layer_count), ULL(h.num_kv_heads), ULL(h.head_dim),
                         ULL(pool->cfg.layer_count), ULL(pool->g.kv_heads), ULL(pool->g.head_dim));
    if (expected_fingerprint &&
        (expected_fingerprint_len != h.fingerprint_len ||
         memcmp(expected_fingerprint, b8 + h.fingerprint_offset, h.fingerprint_len) != 0))
        return set_error(pool->err, ITAK_KV_FINGERPRINT_MISMATCH, "snapshot", 0, 0, 0, 0,
                         "model fingerprint mismatch: need %.*s, snapshot carries %.*s",
                         int(std::min<uint64_t>(expected_fingerprint_len, 400)), expected_fingerprint,
                         int(std::min<uint64_t>(h.fingerprint_len, 400)),
                         reinterpret_cast<const char *>(b8 + h.fingerprint_offset));
    std::vector<itak_snapshot_layer> layers(ls.size());
    const uint8_t *at = rows ? rows - ls[0].keys_offset : b8;
    for (size_t i = 0; i < ls.size(); ++i)
        layers[i] = itak_snapshot_layer{ls[i].first_position, ls[i].rows, at + ls[i].keys_offset,
                                        at + ls[i].values_offset};
    return itak_kv_restore_snapshot(pool, slot, h.token_count, layers.data(), layers.size(),
                                    h.elem ? ITAK_ELEM_F16 : ITAK_ELEM_F32);
}

}  // namespace itak

static itak_status capture_itkv(itak_pool *pool, uint32_t slot, const char *fingerprint,
                                uint64_t fingerprint_len, bool f16_rows, void *out,
                                uint64_t capacity, uint64_t *written, bool with_checksum);

namespace itak {

int32_t capture_itkv_unsummed(itak_pool *pool, uint32_t slot, const char *fingerprint,
                              uint64_t fingerprint_len, bool f16_rows, void *out, uint64_t capacity,
                              uint64_t *written) {
    if (pool && f16_rows && !pool->elem_f16)
        return unsupported(pool->err,
                           "an f16 snapshot of an f32 pool would drop precision the cache holds");
    return capture_itkv(pool, slot, fingerprint, fingerprint_len, f16_rows, out, capacity, written,
                        false);
}

}  // namespace itak

extern "C" {

uint32_t itak_abi_version(void) { return 1; }

const char *itak_last_error(const itak_pool *pool) {
    return pool ? pool->err.message.c_str() : g_create_error.message.c_str();
}

itak_status itak_last_error_info(const itak_pool *pool, itak_error_info *out) {
    if (!out) return ITAK_INVALID_ARGUMENT;
    *out = pool ? pool->err.info : g_create_error.info;
    return ITAK_OK;
}

itak_status itak_pool_create(const itak_pool_config *config, itak_pool **out) {
    ErrorState &e = g_create_error;
    if (!out) return invalid_argument(e, "out is null");
    *out = nullptr;
    if (!config) return invalid_argument(e, "config is null");
    // KvCache::new (cache.rs:327-351) and LayerCache::new (cache.rs:125-141).
    if (config->layer_count == 0) return zero_dimension(e, "layer pattern");
    if (config->num_kv_heads == 0) return zero_dimension(e, "num_kv_heads");
    if (config->head_dim == 0) return zero_dimension(e, "head_dim");
    bool any_windowed = false;
    for (uint32_t i = 0; i < config->layer_count; ++i) {
        if (config->layer_kinds && config->layer_kinds[i] == ITAK_LAYER_WINDOWED) {
            any_windowed = true;
            const uint64_t w = config->windows ? config->windows[i] : 0;
            if (w == 0) return invalid_window(e, 0);
        } else if (config->layer_kinds && config->layer_kinds[i] != ITAK_LAYER_GLOBAL) {
            return invalid_argument(e, "unknown layer kind");
        }
    }
    uint64_t row = 0;
    if (__builtin_mul_overflow(config->num_kv_heads, config->head_dim, &row))
        return size_overflow(e, "kv row length");
    for (uint32_t i = 0; any_windowed && i < config->layer_count; ++i) {
        if (config->layer_kinds[i] != ITAK_LAYER_WINDOWED) continue;
        uint64_t slots = 0;
        if (__builtin_mul_overflow(config->windows[i], row, &slots))  // cache.rs:131-137
            return size_overflow(e, "windowed layer storage");
    }
    if (config->elem != ITAK_ELEM_F32 && config->elem != ITAK_ELEM_F16)
        return invalid_argument(e, "elem is neither ITAK_ELEM_F32 nor ITAK_ELEM_F16");
    if (config->max_slots == 0) return zero_dimension(e, "max_slots");
    if (config->capacity_rows == 0) return zero_dimension(e, "capacity_rows");
    if (config->capacity_rows > (1ull << 30) || config->head_dim > (1u << 16) ||
        config->num_kv_heads > (1u << 16))
        return size_overflow(e, "global layer storage");
    const uint64_t headroom = config->ring_headroom ? config->ring_headroom : 64;
    if (headroom > (1ull << 20)) return size_overflow(e, "windowed layer storage");
    const uint64_t elem_bytes = config->elem == ITAK_ELEM_F16 ? 2 : 4;
    // f16 pools whose head_dim suits the MFMA kernels keep value planes in transposed
    // 32-row blocks; their planes are padded to whole blocks.
    const bool v_blocked = config->elem == ITAK_ELEM_F16 && config->head_dim % 16 == 0;

    // The pattern: global layers share one group of planes, windowed layers another whose
    // planes hold the longest ring. A ring is window + headroom rows rounded up to whole
    // 32-row blocks, so that a 32-position block is also a 32-row block of the ring.
    std::vector<LayerInfo> layers(config->layer_count);
    uint32_t n_global = 0, n_windowed = 0;
    uint64_t max_ring = 0;
    for (uint32_t i = 0; i < config->layer_count; ++i) {
        LayerInfo &L = layers[i];
        L.windowed = config->layer_kinds && config->layer_kinds[i] == ITAK_LAYER_WINDOWED;
        if (!L.windowed) {
            L.index = n_global++;
            continue;
        }
        L.index = n_windowed++;
        L.window = config->windows[i];
        if (L.window > (1ull << 30)) return size_overflow(e, "windowed layer storage");
        L.ring = uint32_t(align_up(L.window + headroom, kVBlock));
        max_ring = std::max<uint64_t>(max_ring, L.ring);
    }
    auto make_geom = [&](uint64_t plane_rows, uint64_t layer_count, PoolGeom &g,
                         uint64_t &bytes) -> bool {
        uint64_t head_stride, side_stride, slot_stride, layer_stride, total;
        if (__builtin_mul_overflow(plane_rows, config->head_dim, &head_stride) ||
            __builtin_mul_overflow(head_stride, config->num_kv_heads, &side_stride) ||
            __builtin_mul_overflow(side_stride, uint64_t(2), &slot_stride) ||
            __builtin_mul_overflow(slot_stride, uint64_t(config->max_slots), &layer_stride) ||
            __builtin_mul_overflow(layer_stride, layer_count, &total) ||
            __builtin_mul_overflow(total, elem_bytes, &bytes))
            return false;
        g.kv_heads = uint32_t(config->num_kv_heads);
        g.head_dim = uint32_t(config->head_dim);
        g.capacity = uint32_t(plane_rows);
        g.max_slots = config->max_slots;
        g.v_block = v_blocked ? kVBlock : 0;
        g.head_stride = head_stride;
        g.side_stride = side_stride;
        g.slot_stride = slot_stride;
        g.layer_stride = layer_stride;
        return true;
    };
    // Planes whose size in bytes is a multiple of 1 MiB + 8 KiB or of 1 MiB - 8 KiB put the
    // streams of a multi-slot launch (one per slot, head and side, a plane apart, all advancing
    // together) onto few memory channels: measured on an MI355X, 32 slots at context 4096 decode
    // in 69 us per layer with planes of 129 blocks of 8 KiB and in 51 us with 128 or 130 (127,
    // 254, 258, 387 and 516 blocks likewise 60 to 66 us against 52). Such a plane gets one more
    // block; the rows are never addressed (a ring's length is its own).
    // The distance between two slots' planes of a head (2 * kv_heads planes) is held to the same
    // rule: that is the spacing of a batch's streams.
    auto spread = [&](uint64_t rows) -> uint64_t {
        const uint64_t step = kVBlock;
        auto bad = [](uint64_t bytes) {
            return bytes != 0 && (bytes % ((1u << 20) + (1u << 13)) == 0 ||
                                  bytes % ((1u << 20) - (1u << 13)) == 0);
        };
        for (int guard = 0; guard < 8; ++guard) {
            const uint64_t plane_bytes = rows * config->head_dim * elem_bytes;
            if (!bad(plane_bytes) && !bad(plane_bytes * 2 * config->num_kv_heads)) break;
            rows += step;
        }
        return rows;
    };
    const uint64_t plane_rows =
        spread(v_blocked ? align_up(config->capacity_rows, kVBlock) : config->capacity_rows);
    PoolGeom g{}, gw{};
    uint64_t bytes_g = 0, bytes_w = 0, bytes = 0;
    if (!make_geom(plane_rows, n_global, g, bytes_g))
        return size_overflow(e, "global layer storage");
    if (!make_geom(spread(max_ring), n_windowed, gw, bytes_w))
        return size_overflow(e, "windowed layer storage");
    bytes_g = align_up(bytes_g, 256);
    if (__builtin_add_overflow(bytes_g, bytes_w, &bytes) || bytes == 0)
        return size_overflow(e, "global layer storage");

    hipError_t he = hipSetDevice(config->device);
    if (he != hipSuccess) return hip_error(e, he, "select device");
    itak_pool *pool = new itak_pool();
    pool->cfg = *config;
    pool->cfg.layer_kinds = nullptr;  // the caller's arrays are not retained: see `layers`
    pool->cfg.windows = nullptr;
    pool->layers = std::move(layers);
    pool->global_layers = n_global;
    pool->windowed_layers = n_windowed;
    pool->headroom = headroom;
    pool->elem_f16 = config->elem == ITAK_ELEM_F16;
    pool->elem_bytes = uint32_t(elem_bytes);
    pool->row = row;
    pool->g = g;
    pool->gw = gw;
    pool->rows_limit = config->capacity_rows;
    pool->bytes = bytes;
    // Rotation frequencies: 64 tables (bases and rotated widths) at the head dims that can attend.
    pool->rope_tables_max = uint32_t(std::clamp<uint64_t>(16384 / config->head_dim, 4, 64));
    const uint64_t tables = pool->rope_tables_max * (config->head_dim / 2) * sizeof(double);
    uint64_t planes = 0, all = 0;
    if (__builtin_add_overflow(bytes, uint64_t(255), &planes) ||
        __builtin_add_overflow(planes &= ~uint64_t(255), tables, &all)) {
        delete pool;
        return size_overflow(e, "global layer storage");
    }
    // They lie behind the planes, unless that takes the planes over the 64 MB up to which the runtime keeps
    // freed memory: 8 layers x 4 KV heads x 4,096 positions, exactly 64 MB, made and freed in 19 + 37 us, with the
    // tables behind them 41 + 270, beside them 20 + 41.
    constexpr uint64_t kKeptByRuntime = 64ull << 20;
    pool->rope_apart = planes <= kKeptByRuntime && all > kKeptByRuntime;
    he = hipMalloc(reinterpret_cast<void **>(&pool->base), pool->rope_apart ? bytes : all);
    if (he != hipSuccess) {
        delete pool;
        return hip_error(e, he, "allocate KV pool");
    }
    pool->base_w = pool->base + bytes_g;
    // Fresh storage is all zero bytes, as the reference's ring storage is
    // (cache.rs:139) and as the scrub guarantee needs.
    he = hipMemset(pool->base, 0, bytes);
    if (he != hipSuccess) {
        (void)hipFree(pool->base);
        delete pool;
        return hip_error(e, he, "zero KV pool");
    }
    pool->slots.resize(config->max_slots);
    pool->ring_saved.assign(config->max_slots, nullptr);
    pool->ring_saved_bytes.assign(config->max_slots, 0);
    pool->merge_in_launch = (config->flags & ITAK_POOL_MERGE_IN_LAUNCH) != 0;
    pool->q_two_halves = pool->elem_f16 && (config->flags & ITAK_POOL_Q_TWO_HALVES) != 0;
    pool->prep_by_launch = (config->flags & ITAK_POOL_PREP_BY_LAUNCH) != 0;
    if (pool->elem_f16 && !pool->merge_in_launch && (config->flags & ITAK_POOL_DIE_MERGE) &&
        die_layout_ok(config->device)) {
        he = hipMalloc(reinterpret_cast<void **>(&pool->die_words), kDieTicketBytes + 256);
        if (he == hipSuccess) he = hipMemset(pool->die_words, 0, kDieTicketBytes + 256);
        if (he != hipSuccess) {
            if (pool->die_words) (void)hipFree(pool->die_words);
            (void)hipFree(pool->base);
            delete pool;
            return hip_error(e, he, "allocate the split tickets");
        }
        pool->die_merge = true;
    }
    he = bind_scratch(config->device, &pool->scratch_dev);
    if (he != hipSuccess) {
        (void)hipFree(pool->base);
        delete pool;
        return hip_error(e, he, "look up the static split workspace");
    }
    pool->rope_dev = reinterpret_cast<double *>(pool->base + planes);
    if (pool->rope_apart && hipMalloc(reinterpret_cast<void **>(&pool->rope_dev), tables) != hipSuccess) {
        (void)hipGetLastError();
        pool->rope_dev = nullptr;
        pool->rope_tables_max = 0;  // (the preparation kernel then takes the powers itself)
    }
    ITAK_DIAG("kv pool built layers=%u kv_heads=%llu head_dim=%llu elem=%s slots=%u capacity_rows=%llu "
              "device_bytes=%llu",
              config->layer_count, ULL(config->num_kv_heads), ULL(config->head_dim),
              pool->elem_f16 ? "f16" : "f32", config->max_slots, ULL(config->capacity_rows),
              ULL(pool->bytes));
    *out = pool;
    return ITAK_OK;
}

void itak_pool_destroy(itak_pool *pool) {
    if (!pool) return;
    (void)hipStreamSynchronize(pool->stream);
    if (pool->base) (void)hipFree(pool->base);
    if (pool->rope_apart && pool->rope_dev) (void)hipFree(pool->rope_dev);
    if (pool->stage) (void)hipFree(pool->stage);
    if (pool->ws) (void)hipFree(pool->ws);
    if (pool->prep) (void)hipFree(pool->prep);
    if (pool->xws) (void)hipFree(pool->xws);
    if (pool->die_words) (void)hipFree(pool->die_words);
    for (void *buf : pool->ring_saved)
        if (buf) (void)hipFree(buf);
    release_hstage(pool);
    pool->ring.close();
    delete pool;
}

itak_status itak_pool_set_stream(itak_pool *pool, void *hip_stream) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    const hipStream_t next = static_cast<hipStream_t>(hip_stream);
    if (next != pool->stream && pool->turns.running()) {
        // A host-pointer call has returned on the arrival of its output, and its last launch may still be
        // storing rows: what the new stream is given must find them. Not where one of the two streams is
        // being captured (a wait would spoil the capture): nothing captured runs before its first replay,
        // and the next host-pointer call waits in any case.
        const hipStream_t tail = stream_of(pool->turns);
        auto idle = [](hipStream_t s) {
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
            return hipStreamIsCapturing(s, &status) == hipSuccess && status == hipStreamCaptureStatusNone;
        };
        if (idle(tail) && idle(next)) {
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // (some other stream of this thread may be captured)
            const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
            if (hipStreamSynchronize(tail) == hipSuccess) pool->turns.drained();
            if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
        }
        (void)hipGetLastError();
    }
    pool->stream = next;
    return ITAK_OK;
}

itak_status itak_pool_synchronize(itak_pool *pool) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize");
    // Consumers of an in-launch merge that gave up waiting counted themselves in their
    // buffer's first word; their outputs are NaN and the buffer may hold words nobody took,
    // so it is made clean again.
    unsigned long long *buffers[2] = {pool->xws,
                                      pool->scratch_exchange_used
                                          ? reinterpret_cast<unsigned long long *>(pool->scratch_dev)
                                          : nullptr};
    const uint64_t words[2] = {pool->xws_words, kScratchExchangeBytes / 8};
    uint32_t total = 0;
    for (int i = 0; i < 2; ++i) {
        if (!buffers[i]) continue;
        uint32_t gave_up = 0;
        HIP_TRY(pool, hipMemcpy(&gave_up, buffers[i], sizeof(gave_up), hipMemcpyDeviceToHost),
                "read the split merge's give-up counter");
        if (!gave_up) continue;
        total += gave_up;
        HIP_TRY(pool, launch_fill_words(buffers[i], words[i], kExchangeEmptyWord, pool->stream),
                "fill the split exchange buffer");
        HIP_TRY(pool, launch_fill_words(buffers[i], 1, 0, pool->stream), "zero the give-up counter");
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize");
    }
    if (total)
        return set_error(pool->err, ITAK_STEP_FAILED, "attention", total, 0, 0, 0,
                         "attention: %u workgroups of a split merge gave up waiting for their "
                         "group; their outputs are NaN and every step launched on this pool since "
                         "the last successful synchronize is invalid",
                         total);
    if (pool->die_words) {
        // A launch that merges on the units' compute dies relies on where the device runs each
        // workgroup; every workgroup checks, and one that ran elsewhere has counted itself.
        uint32_t strays = 0;
        uint32_t *faults = pool->die_words + kDieTicketBytes / sizeof(uint32_t);
        HIP_TRY(pool, hipMemcpy(&strays, faults, sizeof(strays), hipMemcpyDeviceToHost),
                "read the die check's counter");
        if (strays) {
            pool->die_merge = false;  // the ordinary merge launch from here on
            HIP_TRY(pool, hipMemset(pool->die_words, 0, kDieTicketBytes + 256), "clear the split tickets");
            return set_error(pool->err, ITAK_STEP_FAILED, "attention", strays, 0, 0, 0,
                             "attention: %u workgroups of a split merge ran on another compute die "
                             "than their index names; outputs of the steps since the last "
                             "synchronize may be wrong (later steps use the merge launch)",
                             strays);
        }
    }
    return ITAK_OK;
}

itak_status itak_pool_set_merge_spin_limit(itak_pool *pool, uint32_t polls) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    pool->spin_limit = polls;
    return ITAK_OK;
}

uint64_t itak_pool_device_bytes(const itak_pool *pool) { return pool ? pool->bytes : 0; }

itak_status itak_slot_acquire(itak_pool *pool, uint32_t *slot) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!slot) return invalid_argument(pool->err, "slot is null");
    for (uint32_t i = 0; i < pool->slots.size(); ++i) {
        Slot &s = pool->slots[i];
        if (s.in_use) continue;
        s = Slot{};
        s.in_use = true;
        s.cache_id = g_next_cache_id++;
        s.appended.assign(pool->cfg.layer_count, 0);
        s.high.assign(pool->cfg.layer_count, 0);
        s.floor.assign(pool->cfg.layer_count, 0);
        *slot = i;
        return ITAK_OK;
    }
    return set_error(pool->err, ITAK_NO_FREE_SLOT, nullptr, pool->slots.size(), 0, 0, 0,
                     "all %llu slots of the pool are in use", ULL(pool->slots.size()));
}

itak_status itak_slot_reset(itak_pool *pool, uint32_t slot) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    uint64_t max_rows = 0;
    bool ring_used = false;
    for (uint64_t l = 0; l < s->high.size(); ++l) {
        if (pool->layers[l].windowed)
            ring_used = ring_used || s->high[l] > 0;
        else
            max_rows = std::max(max_rows, s->high[l]);
    }
    if (max_rows > 0) {
        ZeroBatch zb{};
        zb.n = 1;
        zb.max_rows = uint32_t(max_rows);
        zb.item[0] = ZeroItem{slot, 0, uint32_t(max_rows), 0};
        itak_status st = scrub_rows(pool, zb);
        if (st != ITAK_OK) return st;
    }
    if (ring_used) {  // the whole ring of every windowed layer
        ZeroBatch zb{};
        zb.n = 1;
        zb.max_rows = pool->gw.capacity;
        zb.item[0] = ZeroItem{slot, 0, pool->gw.capacity, 0};
        HIP_TRY(pool,
                launch_zero_rows(pool->base_w, pool->elem_f16, pool->gw, 0, pool->windowed_layers,
                                 zb, pool->stream),
                "launch ring scrub");
    }
    std::fill(s->appended.begin(), s->appended.end(), 0);
    std::fill(s->high.begin(), s->high.end(), 0);
    std::fill(s->floor.begin(), s->floor.end(), 0);
    s->built = false;
    s->cp = LiveCheckpoint{};
    s->next_serial = 0;
    s->cache_id = g_next_cache_id++;  // outstanding handles go stale (cache.rs:721-728)
    return ITAK_OK;
}

itak_status itak_slot_release(itak_pool *pool, uint32_t slot) {
    itak_status st = itak_slot_reset(pool, slot);
    if (st != ITAK_OK) return st;
    pool->slots[slot].in_use = false;
    return ITAK_OK;
}

uint64_t itak_kv_layer_count(const itak_pool *pool) { return pool ? pool->cfg.layer_count : 0; }
uint64_t itak_kv_num_kv_heads(const itak_pool *pool) { return pool ? pool->g.kv_heads : 0; }
uint64_t itak_kv_head_dim(const itak_pool *pool) { return pool ? pool->g.head_dim : 0; }

itak_status itak_kv_layer_kind(itak_pool *pool, uint64_t layer, uint32_t *kind, uint64_t *window) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (kind) *kind = pool->layers[layer].windowed ? ITAK_LAYER_WINDOWED : ITAK_LAYER_GLOBAL;
    if (window) *window = pool->layers[layer].window;
    return ITAK_OK;
}

itak_status itak_kv_storage_rows(itak_pool *pool, uint64_t layer, uint64_t *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (!out) return invalid_argument(pool->err, "out is null");
    *out = pool->layers[layer].windowed ? pool->layers[layer].ring : pool->rows_limit;
    return ITAK_OK;
}

itak_status itak_kv_stored_len(itak_pool *pool, uint32_t slot, uint64_t layer, uint64_t *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!out) return invalid_argument(pool->err, "out is null");
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    *out = stored_of(pool, *s, layer);  // cache.rs:154-159
    return ITAK_OK;
}

itak_status itak_kv_next_position(itak_pool *pool, uint32_t slot, uint64_t layer, uint64_t *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!out) return invalid_argument(pool->err, "out is null");
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    *out = s->appended[layer];
    return ITAK_OK;
}

itak_status itak_kv_append(itak_pool *pool, uint32_t slot, uint64_t layer, const float *k,
                           uint64_t k_len, const float *v, uint64_t v_len, uint64_t position) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    // cache.rs:430-471, in order.
    if (k_len != pool->row) return shape_mismatch(pool->err, "k", pool->row, k_len);
    if (v_len != pool->row) return shape_mismatch(pool->err, "v", pool->row, v_len);
    if (s->cp.live && layer < pool->cfg.layer_count) {
        const uint64_t limit = s->cp.bases[layer] + s->cp.max_round_tokens;
        if (position >= limit) return range_exceeded(pool->err, layer, position, limit);
    }
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (position != s->appended[layer])
        return out_of_order(pool->err, layer, s->appended[layer], position);
    if (position >= position_limit(pool, layer))
        return capacity_exceeded(pool->err, layer, position + 1, position_limit(pool, layer));
    if (!k || !v) return invalid_argument(pool->err, "k or v is null");
    const uint64_t bytes = pool->row * sizeof(float);
    itak_status st = ensure_stage(pool, 2 * bytes);
    if (st != ITAK_OK) return st;
    float *kd = reinterpret_cast<float *>(pool->stage);
    float *vd = kd + pool->row;
    HIP_TRY(pool, hipMemcpyAsync(kd, k, bytes, hipMemcpyHostToDevice, pool->stream), "upload k");
    HIP_TRY(pool, hipMemcpyAsync(vd, v, bytes, hipMemcpyHostToDevice, pool->stream), "upload v");
    itak_batch_item item{slot, 1};
    st = run_append(pool, layer, &item, 1, kd, vd);
    if (st != ITAK_OK) return st;
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after append");
    return ITAK_OK;
}

itak_status itak_kv_append_device(itak_pool *pool, uint64_t layer, const itak_batch_item *items,
                                  uint32_t item_count, const float *k_dev, const float *v_dev) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (item_count && (!items || !k_dev || !v_dev))
        return invalid_argument(pool->err, "items, k_dev or v_dev is null");
    std::vector<uint64_t> &named = pool->named;
    named.resize(pool->slots.size(), 0);
    const uint64_t number = ++pool->step_number;
    for (uint32_t i = 0; i < item_count; ++i) {
        Slot *s = find_slot(pool, items[i].slot);
        if (!s) return invalid_argument(pool->err, "slot is not in use");
        if (named[items[i].slot] == number) return invalid_argument(pool->err, "slot listed twice in one step");
        named[items[i].slot] = number;
        uint64_t ok = 0;
        itak_status st = check_append_rows(pool, *s, layer, items[i].rows, &ok);
        if (st != ITAK_OK) return st;
        st = check_block_rows(pool, layer, items[i].rows);
        if (st != ITAK_OK) return st;
    }
    return run_append(pool, layer, items, item_count, k_dev, v_dev);
}

static itak_status restore_layers(itak_pool *pool, uint32_t slot, Slot &s,
                                  const itak_snapshot_layer *layers, const uint64_t *layer_ids,
                                  uint64_t count, uint32_t src_elem) {
    if (src_elem != ITAK_ELEM_F32 && src_elem != ITAK_ELEM_F16)
        return invalid_argument(pool->err, "src_elem is neither ITAK_ELEM_F32 nor ITAK_ELEM_F16");
    if (src_elem == ITAK_ELEM_F16 && !pool->elem_f16)
        return unsupported(pool->err, "an f16 snapshot restores only into an f16 pool");
    const uint64_t src_bytes_per_elem = src_elem == ITAK_ELEM_F16 ? 2 : 4;
    // Sources the device cannot read in place are staged through one temporary buffer.
    uint64_t stage_need = 0;
    PtrClassifier kind_of;
    // Rows that all lie in device memory are gathered in stream order, like a device append: the
    // call returns with the gather enqueued. Host memory of either kind is the caller's to free
    // when the call returns, so the call waits for the stream then.
    bool all_device = true;
    for (uint64_t i = 0; i < count; ++i) {
        if (layers[i].rows == 0) continue;
        const uint64_t bytes = layers[i].rows * pool->row * src_bytes_per_elem;
        if (must_stage(kind_of, layers[i].keys, src_bytes_per_elem)) stage_need += align_up(bytes, 256);
        if (must_stage(kind_of, layers[i].values, src_bytes_per_elem)) stage_need += align_up(bytes, 256);
        const void *usable;
        if (kind_of(layers[i].keys, &usable) != PtrKind::Device ||
            kind_of(layers[i].values, &usable) != PtrKind::Device)
            all_device = false;
    }
    unsigned char *temp = nullptr;
    if (stage_need) HIP_TRY(pool, hipMalloc(reinterpret_cast<void **>(&temp), stage_need), "allocate restore staging");
    uint64_t temp_off = 0;
    itak_status st = ITAK_OK;
    std::vector<RingSpan> staged;
    std::vector<const void *> staged_at(2 * count, nullptr);
    for (uint64_t i = 0; i < count && stage_need; ++i) {
        const uint64_t bytes = layers[i].rows * pool->row * src_bytes_per_elem;
        const void *src[2] = {layers[i].keys, layers[i].values};
        for (int side = 0; side < 2 && bytes; ++side)
            if (must_stage(kind_of, src[side], src_bytes_per_elem)) {
                staged.push_back(RingSpan{src[side], temp + temp_off, bytes});
                staged_at[2 * i + side] = temp + temp_off;
                temp_off += align_up(bytes, 256);
            }
    }
    if (hipError_t he = ring_upload(pool->ring, staged, pool->stream); he != hipSuccess) {
        (void)hipStreamSynchronize(pool->stream);
        if (temp) (void)hipFree(temp);
        return hip_error(pool->err, he, "stage snapshot rows");
    }
    // One gather batch per group of planes (global, windowed), launched when it fills up. A
    // windowed layer's rows go to storage rows position % ring: one run, or two when the
    // positions wrap past the end of the ring (session.rs:320-346 states the same split).
    RestoreBatch batch[2] = {};
    batch[0].slot = batch[1].slot = slot;
    // A ring that was filled and then rewound to empty still holds the old rows; a restore
    // that writes fewer rows than the window must find zeros around them, as in a fresh cache.
    for (uint64_t i = 0; i < count; ++i) {
        const uint64_t layer = layer_ids ? layer_ids[i] : i;
        const LayerInfo &info = pool->layers[layer];
        if (!info.windowed || s.high[layer] == 0) continue;
        ZeroBatch zb{};
        zb.n = 1;
        zb.max_rows = info.ring;
        zb.item[0] = ZeroItem{slot, 0, info.ring, 0};
        hipError_t e = launch_zero_rows(pool->base_w, pool->elem_f16, pool->gw, info.index,
                                        info.index + 1, zb, pool->stream);
        if (e != hipSuccess) {
            if (temp) (void)hipFree(temp);
            return hip_error(pool->err, e, "launch ring scrub");
        }
    }
    auto flush = [&](int w) -> itak_status {
        if (batch[w].n == 0) return ITAK_OK;
        hipError_t e = launch_restore(w ? pool->base_w : pool->base, pool->elem_f16,
                                      src_elem == ITAK_ELEM_F16, w ? pool->gw : pool->g, batch[w],
                                      pool->stream);
        batch[w].n = 0;
        batch[w].max_rows = 0;
        return e == hipSuccess ? ITAK_OK : hip_error(pool->err, e, "launch restore gather");
    };
    for (uint64_t i = 0; i < count && st == ITAK_OK; ++i) {
        const itak_snapshot_layer &L = layers[i];
        if (L.rows == 0) continue;
        const uint64_t layer = layer_ids ? layer_ids[i] : i;
        const LayerInfo &info = pool->layers[layer];
        const void *src[2] = {L.keys, L.values};
        for (int side = 0; side < 2; ++side) {
            const void *usable;
            if (staged_at[2 * i + side]) {
                src[side] = staged_at[2 * i + side];
            } else {
                kind_of(src[side], &usable);
                src[side] = usable;
            }
        }
        const int w = info.windowed ? 1 : 0;
        uint64_t done = 0;
        while (done < L.rows && st == ITAK_OK) {
            const uint64_t position = L.first_position + done;
            const uint64_t row = info.windowed ? position % info.ring : position;
            const uint64_t run =
                info.windowed ? std::min<uint64_t>(L.rows - done, info.ring - row) : L.rows - done;
            if (batch[w].n == kMaxRestoreLayers) st = flush(w);
            if (st != ITAK_OK) break;
            RestoreLayer &R = batch[w].layer[batch[w].n++];
            const uint64_t skip = done * pool->row * src_bytes_per_elem;
            R.keys = static_cast<const unsigned char *>(src[0]) + skip;
            R.values = static_cast<const unsigned char *>(src[1]) + skip;
            R.layer = info.index;
            R.rows = uint32_t(run);
            R.first_row = uint32_t(row);
            batch[w].max_rows = std::max(batch[w].max_rows, R.rows);
            done += run;
        }
    }
    for (int w = 0; w < 2 && st == ITAK_OK; ++w) st = flush(w);
    if (!all_device || stage_need || st != ITAK_OK) {
        hipError_t he = hipStreamSynchronize(pool->stream);
        if (st == ITAK_OK && he != hipSuccess) st = hip_error(pool->err, he, "synchronize after restore");
    }
    if (temp) (void)hipFree(temp);
    if (st != ITAK_OK) return st;
    for (uint64_t i = 0; i < count; ++i) {
        const uint64_t layer = layer_ids ? layer_ids[i] : i;
        s.appended[layer] = layers[i].first_position + layers[i].rows;  // cache.rs:568
        s.high[layer] = s.appended[layer];
        s.floor[layer] = layers[i].first_position;
        ITAK_DIAG("bulk restore slot=%u layer=%llu first_position=%llu rows=%llu appended=%llu", slot,
                  ULL(layer), ULL(layers[i].first_position), ULL(layers[i].rows),
                  ULL(s.appended[layer]));
    }
    return ITAK_OK;
}

itak_status itak_kv_restore_bulk(itak_pool *pool, uint32_t slot, uint64_t layer,
                                 uint64_t first_position, const void *keys, uint64_t keys_len,
                                 const void *values, uint64_t values_len, uint32_t src_elem) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    // cache.rs:520-546, in order.
    if (keys_len != values_len || keys_len % pool->row != 0)
        return shape_mismatch(pool->err, "bulk restore rows", values_len, keys_len);
    const uint64_t rows = keys_len / pool->row;
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (s->appended[layer] != 0) return not_fresh(pool->err, layer, s->appended[layer]);
    if (pool->layers[layer].windowed) {
        if (rows > pool->layers[layer].window)
            return shape_mismatch(pool->err, "bulk restore rows (windowed layer)",
                                  pool->layers[layer].window, rows);
    } else if (first_position != 0) {
        return shape_mismatch(pool->err, "bulk restore first position (global layer)", 0,
                              first_position);
    }
    if (first_position > position_limit(pool, layer) ||
        rows > position_limit(pool, layer) - first_position)
        return capacity_exceeded(pool->err, layer, first_position + rows,
                                 position_limit(pool, layer));
    if (rows && (!keys || !values)) return invalid_argument(pool->err, "keys or values is null");
    itak_snapshot_layer L{first_position, rows, keys, values};
    return restore_layers(pool, slot, *s, &L, &layer, 1, src_elem);
}

itak_status itak_kv_restore_snapshot(itak_pool *pool, uint32_t slot, uint64_t token_count,
                                     const itak_snapshot_layer *layers, uint64_t layer_count,
                                     uint32_t src_elem) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!layers) return invalid_argument(pool->err, "layers is null");
    // KvSnapshot::validate (snapshot.rs:187-236) against the pool's own pattern.
    if (layer_count != pool->cfg.layer_count)
        return set_error(pool->err, ITAK_STEP_FAILED, "restore_snapshot", layer_count,
                         pool->cfg.layer_count, 0, 0,
                         "snapshot carries %llu layer blocks but its geometry has %llu layers",
                         ULL(layer_count), ULL(pool->cfg.layer_count));
    for (uint64_t i = 0; i < layer_count; ++i) {
        const LayerInfo &info = pool->layers[i];
        const uint64_t expected_rows =
            info.windowed ? std::min(token_count, info.window) : token_count;
        const uint64_t expected_first = token_count - expected_rows;
        if (layers[i].first_position != expected_first) {
            char kind[64] = "Global";
            if (info.windowed)
                snprintf(kind, sizeof(kind), "Windowed { window: %llu }", ULL(info.window));
            return set_error(pool->err, ITAK_STEP_FAILED, "restore_snapshot", i,
                             layers[i].first_position, expected_first, 0,
                             "layer %llu: first stored position is %llu but %llu follows from token "
                             "count %llu and kind %s",
                             ULL(i), ULL(layers[i].first_position), ULL(expected_first),
                             ULL(token_count), kind);
        }
        if (layers[i].rows != expected_rows)
            return set_error(pool->err, ITAK_STEP_FAILED, "restore_snapshot", i, layers[i].rows,
                             expected_rows, 0,
                             "layer %llu: holds %llu rows but %llu rows were expected", ULL(i),
                             ULL(layers[i].rows), ULL(expected_rows));
        if (expected_rows && (!layers[i].keys || !layers[i].values))
            return invalid_argument(pool->err, "a layer's keys or values is null");
    }
    // KvSnapshot::restore builds a fresh cache (snapshot.rs:321-334): every layer must be
    // fresh here, checked for all layers before any is touched.
    for (uint64_t i = 0; i < layer_count; ++i)
        if (s->appended[i] != 0) return not_fresh(pool->err, i, s->appended[i]);
    for (uint64_t i = 0; i < layer_count; ++i)
        if (token_count > position_limit(pool, i))
            return capacity_exceeded(pool->err, i, token_count, position_limit(pool, i));
    return restore_layers(pool, slot, *s, layers, nullptr, layer_count, src_elem);
}

// ---- itak_kv: hashes, the ITKV codec, capture and restore of encoded snapshots ----------

uint64_t itak_kv_prefix_hash(const uint32_t *tokens, uint64_t count) {  // hash.rs:44-46
    return fnv1a64_tokens(tokens, tokens ? count : 0, kFnvOffset);
}
uint64_t itak_kv_prefix_discriminator(const uint32_t *tokens, uint64_t count) {  // hash.rs:52-54
    return fnv1a64_tokens(tokens, tokens ? count : 0, kFnvAltOffset);
}
uint64_t itak_kv_checksum(const void *bytes, uint64_t count) {  // hash.rs:59-61
    return fnv1a64(static_cast<const uint8_t *>(bytes), bytes ? count : 0, kFnvOffset);
}
uint64_t itak_kv_checksum_blocks(const void *bytes, uint64_t count) {
    return fnv1a64_blocks(static_cast<const uint8_t *>(bytes), bytes ? count : 0);
}

itak_status itak_itkv_validate(const itak_itkv_header *header, const itak_itkv_layer *layers,
                               uint64_t blocks, const uint64_t *key_floats,
                               const uint64_t *value_floats) {
    ErrorState &e = g_create_error;
    if (!header || (blocks && (!layers || !key_floats || !value_floats)))
        return invalid_argument(e, "header, layers or the float counts are null");
    ItkvError err;
    const std::vector<ItkvLayer> ls = to_internal(layers, blocks);
    if (!itkv_validate(to_internal(*header), ls.data(), blocks, key_floats, value_floats, err))
        return set_itkv_error(e, err);
    return ITAK_OK;
}

itak_status itak_itkv_encode(const itak_itkv_header *header, const char *fingerprint,
                             const itak_itkv_layer *layers, uint64_t blocks,
                             const float *const *keys, const uint64_t *key_floats,
                             const float *const *values, const uint64_t *value_floats, void *out,
                             uint64_t capacity, uint64_t *written) {
    ErrorState &e = g_create_error;
    itak_status st = itak_itkv_validate(header, layers, blocks, key_floats, value_floats);
    if (st != ITAK_OK) return st;
    if (!written) return invalid_argument(e, "written is null");
    if (header->fingerprint_len && !fingerprint) return invalid_argument(e, "fingerprint is null");
    if (header->version > 1 || header->elem != 0)
        return unsupported(e, "itak_itkv_encode writes version 1 (f32 rows); version 2 comes from "
                              "itak_kv_capture_itkv_f16");
    if (header->num_kv_heads > UINT32_MAX || header->head_dim > UINT32_MAX ||
        header->layer_count > UINT32_MAX || header->fingerprint_len > UINT32_MAX)
        return invalid_argument(e, "a header field does not fit the 32-bit wire field");
    ItkvHeader h = to_internal(*header);
    std::vector<ItkvLayer> ls = to_internal(layers, blocks);
    uint64_t total = 0;
    if (!itkv_encoded_len(h, ls.data(), &total)) return size_overflow(e, "encoded snapshot");
    *written = total;
    if (!out) return ITAK_OK;
    if (capacity < total) return invalid_argument(e, "output buffer is smaller than the encoding");
    uint8_t *bytes = static_cast<uint8_t *>(out);
    itkv_write_header(bytes, h, fingerprint, ls.data());
    for (uint64_t i = 0; i < blocks; ++i) {
        if (key_floats[i] && (!keys || !keys[i] || !values || !values[i]))
            return invalid_argument(e, "a layer's keys or values is null");
        if (key_floats[i]) {  // f32 little-endian is this host's own representation
            memcpy(bytes + ls[i].keys_offset, keys[i], key_floats[i] * 4);
            memcpy(bytes + ls[i].values_offset, values[i], value_floats[i] * 4);
        }
    }
    const uint64_t sum = fnv1a64(bytes, total - 8, kFnvOffset);
    for (int b = 0; b < 8; ++b) bytes[total - 8 + b] = uint8_t(sum >> (8 * b));
    return ITAK_OK;
}

itak_status itak_itkv_decode(const void *bytes, uint64_t len, itak_itkv_header *header,
                             itak_itkv_layer *layers, uint64_t layers_capacity) {
    ErrorState &e = g_create_error;
    if (!bytes || !header) return invalid_argument(e, "bytes or header is null");
    ItkvHeader h;
    std::vector<ItkvLayer> ls;
    ItkvError err;
    if (!itkv_decode(static_cast<const uint8_t *>(bytes), len, h, ls, err))
        return set_itkv_error(e, err);
    *header = itak_itkv_header{h.token_count,     h.num_kv_heads,       h.head_dim,      h.layer_count,
                               h.fingerprint_len, h.fingerprint_offset, h.encoded_len,   h.version,
                               h.elem};
    if (layers_capacity < ls.size())
        return invalid_argument(e, "layers_capacity is smaller than the snapshot's layer count");
    for (size_t i = 0; i < ls.size(); ++i)
        layers[i] = itak_itkv_layer{ls[i].kind, 0, ls[i].window, ls[i].first_position, ls[i].rows,
                                    ls[i].keys_offset, ls[i].values_offset};
    return ITAK_OK;
}

static itak_status capture_itkv(itak_pool *pool, uint32_t slot, const char *fingerprint,
                                uint64_t fingerprint_len, bool f16_rows, void *out,
                                uint64_t capacity, uint64_t *written, bool with_checksum = true);

itak_status itak_kv_capture_itkv(itak_pool *pool, uint32_t slot, const char *fingerprint,
                                 uint64_t fingerprint_len, void *out, uint64_t capacity,
                                 uint64_t *written) {
    return capture_itkv(pool, slot, fingerprint, fingerprint_len, false, out, capacity, written);
}

itak_status itak_kv_capture_itkv_f16(itak_pool *pool, uint32_t slot, const char *fingerprint,
                                     uint64_t fingerprint_len, void *out, uint64_t capacity,
                                     uint64_t *written) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!pool->elem_f16)
        return unsupported(pool->err,
                           "an f16 snapshot of an f32 pool would drop precision the cache holds");
    return capture_itkv(pool, slot, fingerprint, fingerprint_len, true, out, capacity, written);
}

// A snapshot's payload passes through device memory this many bytes at a time (a multiple of the
// ring's chunk and of the hash's runs). From kDeviceSumBytes on the checksum is the
// device's: its six launches take 30 us there, what a host core needs for 36 KiB, and the rule
// leaves a margin for their coming one behind the other on a busy stream. (Version 2's was
// the host threads' until its blocks' sums came to the device: fnv_kernels.hip.)
constexpr uint64_t kPayloadPiece = 32ull << 20;
constexpr uint64_t kDeviceSumBytes = 128ull << 10;
static_assert(kPayloadPiece == kRingChunk * kRingSlots && kRingChunk % kFnvRun == 0, "pieces are whole chunks and runs");

// A large output buffer is often fresh from the allocator: its pages are touched here for the
// first time, and 4 KiB at a time that costs more than the copy. Only a hint; a refusal is no loss.
static void advise_huge_pages(void *p, uint64_t bytes) {
    const uint64_t huge = 2ull << 20;
    const uint64_t from = align_up(reinterpret_cast<uint64_t>(p), huge), to = (reinterpret_cast<uint64_t>(p) + bytes) / huge * huge;
    if (to > from && to - from >= 4 * huge) (void)madvise(reinterpret_cast<void *>(from), to - from, MADV_HUGEPAGE);
}

// Version 2's block sums can be made on the device where the header ends in the first block.
static uint64_t sum_blocks(uint64_t file_bytes) { return (file_bytes + kItkvSumBlock - 1) / kItkvSumBlock; }
static bool device_sums(uint32_t version, uint64_t payload_at) { return version == kItkvVersion || payload_at < kItkvSumBlock; }

static itak_status finish_capture(uint8_t *bytes, uint64_t total, uint32_t version, bool with_checksum,
                                  const uint64_t *known) {
    const uint64_t sum = known ? *known : with_checksum ? itkv_trailer(version, bytes, total - 8) : 0;
    for (int b = 0; b < 8; ++b) bytes[total - 8 + b] = uint8_t(sum >> (8 * b));
    return ITAK_OK;
}

static itak_status capture_itkv(itak_pool *pool, uint32_t slot, const char *fingerprint,
                                uint64_t fingerprint_len, bool f16_rows, void *out,
                                uint64_t capacity, uint64_t *written, bool with_checksum) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!written) return invalid_argument(pool->err, "written is null");
    if (fingerprint_len && !fingerprint) return invalid_argument(pool->err, "fingerprint is null");
    if (fingerprint_len > UINT32_MAX) return invalid_argument(pool->err, "fingerprint too long");
    // snapshot.rs:249-262: one sequence, every layer at the same position.
    const uint64_t token_count = s->appended[0];
    for (uint64_t i = 0; i < pool->cfg.layer_count; ++i)
        if (s->appended[i] != token_count)
            return set_error(pool->err, ITAK_KV_INCOHERENT_CACHE, "snapshot", token_count,
                             s->appended[i], i, 0,
                             "incoherent cache: layer 0 has appended %llu positions but layer %llu "
                             "has appended %llu; a snapshot is one sequence",
                             ULL(token_count), ULL(i), ULL(s->appended[i]));
    ItkvHeader h;
    h.token_count = token_count;
    h.num_kv_heads = pool->g.kv_heads;
    h.head_dim = pool->g.head_dim;
    h.layer_count = pool->cfg.layer_count;
    h.fingerprint_len = fingerprint_len;
    if (f16_rows) {
        h.version = kItkvVersionTyped;
        h.elem = ITAK_ELEM_F16;
    }
    const uint64_t out_elem = h.elem_bytes();
    // snapshot.rs:264-295: every row of a global layer, the last `window` rows of a windowed
    // one, oldest first.
    std::vector<ItkvLayer> ls(h.layer_count);
    for (uint64_t i = 0; i < h.layer_count; ++i) {
        const LayerInfo &info = pool->layers[i];
        ls[i].kind = info.windowed ? ITAK_LAYER_WINDOWED : ITAK_LAYER_GLOBAL;
        ls[i].window = info.window;
        ls[i].rows = stored_of(pool, *s, i);
        ls[i].first_position = token_count - ls[i].rows;
    }
    uint64_t total = 0;
    if (!itkv_encoded_len(h, ls.data(), &total)) return size_overflow(pool->err, "encoded snapshot");
    *written = total;
    if (!out) return ITAK_OK;
    if (capacity < total)
        return invalid_argument(pool->err, "output buffer is smaller than the encoding");
    uint8_t *bytes = static_cast<uint8_t *>(out);
    itkv_write_header(bytes, h, fingerprint, ls.data());
    if (token_count == 0) return finish_capture(bytes, total, h.version, with_checksum, nullptr);
    // The payload (every layer's keys, then its values) is made in device memory 32 MiB at a time,
    // summed there from kDeviceSumBytes on (version 1's chain, or version 2's blocks), and goes out through the pinned ring.
    const uint64_t payload = ls[0].keys_offset, payload_bytes = total - 8 - payload;
    const uint64_t piece = std::min(align_up(payload_bytes, 256), kPayloadPiece);
    const bool device_sum = with_checksum && payload_bytes >= kDeviceSumBytes && device_sums(h.version, payload);
    const uint64_t blocks = device_sum && h.version != kItkvVersion ? sum_blocks(total - 8) : 0;
    // f32 rows of an f16 pool cross the link as the halves they are and are widened by the host threads that
    // empty the ring (16 layers of 2,000 rows: 4.0 -> 3.05 ms); the sum is over f32 rows made beside them.
    const bool widen = !f16_rows && pool->elem_f16 && host_has_f16();
    const uint64_t halves_bytes = widen ? align_up(piece / 2, 256) : 0;
    const uint64_t scratch_bytes = device_sum ? fnv_scratch_bytes(piece) : 0;
    itak_status st = ensure_stage(pool, piece + 256 + halves_bytes + scratch_bytes + blocks * 8);
    if (st != ITAK_OK) return st;
    unsigned char *rows_dev = pool->stage + 256, *halves_dev = rows_dev + piece, *scratch = halves_dev + halves_bytes;
    // (Version 1's one chain, or version 2's of each block.)
    unsigned long long *state = reinterpret_cast<unsigned long long *>(blocks ? scratch + scratch_bytes : pool->stage);
    advise_huge_pages(bytes, total);
    if (device_sum)
        HIP_TRY(pool, launch_fill_words(state, 1, fnv1a64(bytes, payload, kFnvOffset), pool->stream), "start checksum");
    uint64_t run = 0, run_at = 0;  // the (layer, side) the next byte belongs to, and the first byte of it
    auto make_piece = [&](uint64_t at, uint64_t bytes_here) -> hipError_t {
        ReadRuns b{};
        b.slot = slot;
        const uint64_t end = at + bytes_here;
        for (uint64_t to = at; to < end;) {
            const ItkvLayer &L = ls[run / 2];
            const LayerInfo &info = pool->layers[run / 2];
            const uint64_t run_bytes = L.rows * pool->row * out_elem;
            const uint64_t n = std::min(end, run_at + run_bytes) - to;
            if (n) {
                b.run[b.n++] = ReadRun{info.index, uint32_t(run & 1), uint32_t(L.first_position),
                                       info.windowed ? uint32_t(info.ring) : 0, (to - run_at) / out_elem, n / out_elem,
                                       (to - at) / out_elem};
                to += n;
            }
            if (to == run_at + run_bytes) {
                run_at += run_bytes;
                ++run;
            }
            if (b.n == kMaxReadRuns || to == end) {
                hipError_t e = hipSuccess;
                if (widen)
                    e = launch_read_runs(pool->base, pool->base_w, pool->elem_f16, 1, pool->g, pool->gw, b, halves_dev, pool->stream);
                if (e == hipSuccess && (!widen || device_sum))
                    e = launch_read_runs(pool->base, pool->base_w, pool->elem_f16, f16_rows, pool->g, pool->gw, b, rows_dev,
                                         pool->stream);
                if (e != hipSuccess) return e;
                b.n = 0;
            }
        }
        if (!device_sum) return hipSuccess;
        return blocks ? launch_fnv_blocks(rows_dev, bytes_here, payload + at, scratch, state, pool->stream)
                      : launch_fnv(rows_dev, bytes_here / kFnvRun * kFnvRun, scratch, state, pool->stream);
    };
    HIP_TRY(pool,
            ring_download(pool->ring, bytes + payload, payload_bytes, pool->stream, widen,
                          [&](uint64_t at, uint64_t, const void **src) -> hipError_t {
                              *src = widen ? halves_dev + at % kPayloadPiece / 2 : rows_dev + at % kPayloadPiece;
                              if (at % kPayloadPiece) return hipSuccess;
                              return make_piece(at, std::min(kPayloadPiece, payload_bytes - at));
                          }),
            "download snapshot rows");
    if (!device_sum) return finish_capture(bytes, total, h.version, with_checksum, nullptr);
    std::vector<uint64_t> sums(std::max<uint64_t>(blocks, 1));
    HIP_TRY(pool, hipMemcpyAsync(sums.data(), state, sums.size() * 8, hipMemcpyDeviceToHost, pool->stream), "download checksum");
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after readback");
    uint64_t sum = sums[0];
    if (blocks) {
        sum = fnv1a64_of_sums(sums.data(), blocks);
        return finish_capture(bytes, total, h.version, true, &sum);
    }
    const uint64_t tail = payload_bytes % kFnvRun;  // only the last piece can have one
    sum = fnv1a64(bytes + total - 8 - tail, tail, sum);
    return finish_capture(bytes, total, h.version, true, &sum);
}

// Device memory for the length of a call; freeing it waits for what the call enqueued.
struct DeviceBuffer {
    unsigned char *p = nullptr;
    hipError_t make(uint64_t bytes) {
        const hipError_t e = hipMalloc(reinterpret_cast<void **>(&p), bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
        }
        return e;
    }
    ~DeviceBuffer() {
        if (p) (void)hipFree(p);
    }
};

itak_status itak_kv_restore_itkv(itak_pool *pool, uint32_t slot, const void *bytes, uint64_t len,
                                 const char *expected_fingerprint,
                                 uint64_t expected_fingerprint_len) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!bytes) return invalid_argument(pool->err, "bytes is null");
    // The decoder walks the bytes on the host (header fields, then the checksum over all of
    // them); a device-resident buffer would have to be copied first.
    const void *unused;
    const PtrKind kind = classify(bytes, &unused);
    if (kind == PtrKind::Device)
        return invalid_argument(pool->err, "an encoded snapshot is decoded on the host: pass host memory");
    ItkvHeader h;
    std::vector<ItkvLayer> ls;
    ItkvError err;
    const uint8_t *b8 = static_cast<const uint8_t *>(bytes);
    // From kDeviceSumBytes on the payload goes to the device first, is summed there, and is gathered from there
    // once the sum is known good.
    DeviceBuffer rows;
    hipError_t moved = hipSuccess;
    const ItkvSum sum_of = [&](const ItkvHeader &header, uint64_t payload) -> uint64_t {
        const uint64_t n = len - 8 - payload, piece = std::min(align_up(n, 256), kPayloadPiece);
        const bool device_sum = device_sums(header.version, payload);
        const uint64_t blocks = header.version != kItkvVersion && device_sum ? sum_blocks(len - 8) : 0;
        const uint64_t scratch_bytes = device_sum ? fnv_scratch_bytes(piece) : 0;
        // Rows that an f16 pool wrote are halves again on their way over the link (ring_upload_narrow), and
        // f32 in device memory as the sum and the gather want them (16 layers of 2,000 rows: 3.9 -> 2.7 ms).
        const bool pinned = kind == PtrKind::PinnedHost;
        // (Below, the narrowing and the device's launch take longer than the bytes saved: 1.9 MB 231 us as f32, 249
        // as halves, 4 MB 333 and 311.)
        constexpr uint64_t kNarrowBytes = 3ull << 20;
        LoadRoom room;
        if (n < kDeviceSumBytes ||
            !take_load_room(n, piece, scratch_bytes + blocks * 8,
                            header.version == kItkvVersion && pool->elem_f16 && !pinned && n >= kNarrowBytes && host_has_f16(),
                            [&](uint64_t want) { return rows.make(want) == hipSuccess; }, room))
            return itkv_trailer(header.version, b8, len - 8);
        const bool narrow = room.halves_bytes != 0;
        unsigned long long *state = reinterpret_cast<unsigned long long *>(
            rows.p + (blocks ? room.scratch_at + scratch_bytes : room.state_at));
        if (device_sum)
            moved = launch_fill_words(state, 1, fnv1a64(b8, payload, kFnvOffset), pool->stream);
        uint64_t summed = 0;
        const auto sum_up_to = [&](uint64_t sent) -> hipError_t {
            if (!device_sum || (sent < n && sent - summed < kPayloadPiece)) return hipSuccess;
            unsigned char *scratch = rows.p + room.scratch_at;
            hipError_t e = blocks ? launch_fnv_blocks(rows.p + summed, sent - summed, payload + summed, scratch, state, pool->stream)
                                  : launch_fnv(rows.p + summed, (sent - summed) / kFnvRun * kFnvRun, scratch, state, pool->stream);
            summed = sent;
            return e;
        };
        if (moved == hipSuccess && pinned) {
            for (uint64_t at = 0; at < n && moved == hipSuccess; at += kPayloadPiece) {
                const uint64_t here = std::min(kPayloadPiece, n - at);
                moved = hipMemcpyAsync(rows.p + at, b8 + payload + at, here, hipMemcpyHostToDevice, pool->stream);
                if (moved == hipSuccess) moved = sum_up_to(at + here);
            }
        } else if (moved == hipSuccess && narrow) {
            moved = ring_upload_narrow(pool->ring, b8 + payload, n, rows.p, rows.p + room.halves_at, pool->stream,
                                       [&](uint64_t sent, uint64_t from, uint64_t to) -> hipError_t {
                                           hipError_t e = launch_widen_f16(reinterpret_cast<uint16_t *>(rows.p + room.halves_at + from % kPayloadPiece / 2),
                                                                           reinterpret_cast<float *>(rows.p + from), (to - from) / 4,
                                                                           pool->stream);
                                           return e == hipSuccess && (sent == n || sent % kPayloadPiece == 0) ? sum_up_to(sent) : e;
                                       });
        } else if (moved == hipSuccess) {
            moved = ring_upload(pool->ring, {RingSpan{b8 + payload, rows.p, n}}, pool->stream, sum_up_to);
        }
        std::vector<uint64_t> sums(std::max<uint64_t>(blocks, 1));
        if (!device_sum) sums[0] = itkv_trailer(header.version, b8, len - 8);
        if (moved == hipSuccess && device_sum)
            moved = hipMemcpyAsync(sums.data(), state, sums.size() * 8, hipMemcpyDeviceToHost, pool->stream);
        const hipError_t done = hipStreamSynchronize(pool->stream);
        if (moved == hipSuccess) moved = done;
        if (blocks) return fnv1a64_of_sums(sums.data(), blocks);
        return device_sum ? fnv1a64(b8 + len - 8 - n % kFnvRun, n % kFnvRun, sums[0]) : sums[0];
    };
    const bool decoded = itkv_decode(b8, len, h, ls, err, nullptr, sum_of);
    if (moved != hipSuccess) return hip_error(pool->err, moved, "move snapshot rows to the device");
    if (!decoded) return set_itkv_error(pool->err, err);
    return restore_decoded_itkv(pool, slot, b8, h, ls, expected_fingerprint, expected_fingerprint_len, rows.p);
}

itak_status itak_kv_stats(itak_pool *pool, uint32_t slot, itak_layer_stats *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!out) return invalid_argument(pool->err, "out is null");
    for (uint32_t i = 0; i < pool->cfg.layer_count; ++i) {
        const LayerInfo &info = pool->layers[i];
        out[i] = itak_layer_stats{i, uint32_t(info.windowed ? ITAK_LAYER_WINDOWED : ITAK_LAYER_GLOBAL),
                                  0, info.window, s->appended[i], stored_of(pool, *s, i)};
    }
    return ITAK_OK;
}

// `first` is a position (a storage row on a global layer, which is the same thing); `ring`
// maps positions to storage rows on a windowed layer, 0 reads storage rows as they lie.
static itak_status read_rows_common(itak_pool *pool, uint32_t slot, uint64_t layer, uint64_t first,
                                    uint64_t rows, uint32_t ring, void *keys_out,
                                    void *values_out) {
    if (rows == 0 || (!keys_out && !values_out)) return ITAK_OK;
    const uint64_t bytes = rows * pool->row * pool->elem_bytes;
    itak_status st = ensure_stage(pool, 2 * align_up(bytes, 256));
    if (st != ITAK_OK) return st;
    void *kd = keys_out ? pool->stage : nullptr;
    void *vd = values_out ? pool->stage + align_up(bytes, 256) : nullptr;
    HIP_TRY(pool,
            launch_read_rows(layer_base(pool, layer), pool->elem_f16, geom_of(pool, layer), slot,
                             uint32_t(first), uint32_t(rows), ring, kd, vd, pool->stream),
            "launch row readback");
    if (keys_out)
        HIP_TRY(pool, hipMemcpyAsync(keys_out, kd, bytes, hipMemcpyDeviceToHost, pool->stream),
                "download keys");
    if (values_out)
        HIP_TRY(pool, hipMemcpyAsync(values_out, vd, bytes, hipMemcpyDeviceToHost, pool->stream),
                "download values");
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after readback");
    return ITAK_OK;
}

itak_status itak_kv_read_rows(itak_pool *pool, uint32_t slot, uint64_t layer, uint64_t first,
                              uint64_t rows, void *keys_out, void *values_out,
                              uint64_t *positions_out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    const uint64_t stored = stored_of(pool, *s, layer);
    if (first > stored || rows > stored - first)
        return shape_mismatch(pool->err, "visible rows", stored,
                              rows > UINT64_MAX - first ? UINT64_MAX : first + rows);  // (no wrapped sum in the text)
    const uint64_t oldest = first_visible(pool, *s, layer);
    if (positions_out)
        for (uint64_t i = 0; i < rows; ++i) positions_out[i] = oldest + first + i;  // cache.rs:878-883
    return read_rows_common(pool, slot, layer, oldest + first, rows, pool->layers[layer].ring,
                            keys_out, values_out);
}

itak_status itak_kv_read_raw(itak_pool *pool, uint32_t slot, uint64_t layer, void *keys_out,
                             void *values_out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    const uint64_t rows = pool->layers[layer].windowed ? pool->layers[layer].ring : pool->rows_limit;
    return read_rows_common(pool, slot, layer, 0, rows, 0, keys_out, values_out);
}

// Moves ring rows of the layers in `saves` between their rings and the slot's side buffer:
// positions [from, to) of each layer that fall inside what its save covers.
static itak_status move_ring_rows(itak_pool *pool, uint32_t slot, const Slot &s,
                                  const std::vector<RingSave> &saves, const uint64_t *bases,
                                  uint64_t from, const uint64_t *to_per_layer, bool to_ring) {
    RingRowsBatch b{};
    b.slot = slot;
    auto flush = [&]() -> itak_status {
        if (b.n == 0) return ITAK_OK;
        hipError_t e = launch_ring_rows(pool->base_w, pool->elem_f16, pool->gw, b,
                                        pool->ring_saved[slot], to_ring, pool->stream);
        b.n = 0;
        b.max_rows = 0;
        return e == hipSuccess ? ITAK_OK : hip_error(pool->err, e, "launch ring row copy");
    };
    (void)s;
    for (const RingSave &rs : saves) {
        const uint64_t base = bases[rs.layer];
        const uint64_t lo = std::max(from, base);
        const uint64_t hi = std::min<uint64_t>(to_per_layer[rs.layer], base + rs.rows);
        if (hi <= lo) continue;
        const LayerInfo &L = pool->layers[rs.layer];
        RingRowsLayer &R = b.layer[b.n++];
        R.layer = L.index;
        R.ring = L.ring;
        R.pos0 = uint32_t(lo);
        R.rows = uint32_t(hi - lo);
        R.saved_row0 = uint32_t(lo - base);
        R.saved_rows = rs.rows;
        R.saved_off = rs.saved_off;
        b.max_rows = std::max(b.max_rows, R.rows);
        if (b.n == kMaxRestoreLayers) {
            itak_status st = flush();
            if (st != ITAK_OK) return st;
        }
    }
    return flush();
}

// The checkpoint's copy of the rows a deep round may overwrite (cache.rs:678-697).
static itak_status save_ring_rows(itak_pool *pool, uint32_t slot, const Slot &s,
                                  const std::vector<RingSave> &saves, uint64_t elems) {
    const uint64_t bytes = elems * pool->elem_bytes;
    if (bytes > pool->ring_saved_bytes[slot]) {
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize before growing the checkpoint buffer");
        if (pool->ring_saved[slot]) HIP_TRY(pool, hipFree(pool->ring_saved[slot]), "free the checkpoint buffer");
        pool->ring_saved[slot] = nullptr;
        pool->ring_saved_bytes[slot] = 0;
        HIP_TRY(pool, hipMalloc(&pool->ring_saved[slot], bytes), "allocate the checkpoint buffer");
        pool->ring_saved_bytes[slot] = bytes;
    }
    std::vector<uint64_t> to(pool->layers.size());
    for (const RingSave &rs : saves) to[rs.layer] = s.appended[rs.layer] + rs.rows;
    return move_ring_rows(pool, slot, s, saves, s.appended.data(), 0, to.data(), false);
}

itak_status itak_kv_checkpoint_active(itak_pool *pool, uint32_t slot, int32_t *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!out) return invalid_argument(pool->err, "out is null");
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    *out = s->cp.live ? 1 : 0;
    return ITAK_OK;
}

itak_status itak_kv_checkpoint(itak_pool *pool, uint32_t slot, uint64_t max_round_tokens,
                               itak_checkpoint *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!out) return invalid_argument(pool->err, "out is null");
    // cache.rs:635-651, in order.
    if (s->cp.live) return checkpoint_busy(pool->err);
    if (max_round_tokens == 0) return zero_dimension(pool->err, "max_round_tokens");
    uint64_t smallest_window = 0, windowed = 0;
    for (const LayerInfo &L : pool->layers)
        if (L.windowed) {
            smallest_window = windowed ? std::min(smallest_window, L.window) : L.window;
            ++windowed;
        }
    if (windowed && max_round_tokens > smallest_window)
        return set_error(pool->err, ITAK_CHECKPOINT_TOO_DEEP, nullptr, max_round_tokens,
                         smallest_window, 0, 0,
                         "checkpoint round bound %llu exceeds the smallest sliding window %llu: a "
                         "round that long would overwrite a ring slot twice and no rewind could be "
                         "exact",
                         ULL(max_round_tokens), ULL(smallest_window));
    // A round the ring's headroom covers needs no copies: the rows it overwrites are outside
    // every window a rewind can bring back. A longer one (up to the smallest window, as the
    // reference allows) sets the rows it may overwrite aside first, layer by layer where the
    // headroom is too short, exactly the slots the reference saves (cache.rs:678-697).
    std::vector<RingSave> saves;
    uint64_t save_elems = 0;
    for (uint64_t li = 0; li < pool->layers.size(); ++li) {
        const LayerInfo &L = pool->layers[li];
        if (!L.windowed || max_round_tokens <= L.ring - L.window) continue;
        RingSave rs;
        rs.layer = uint32_t(li);
        rs.rows = uint32_t(max_round_tokens);
        rs.saved_off = save_elems;
        rs.high0 = s->high[li];
        save_elems += 2 * max_round_tokens * pool->row;
        saves.push_back(rs);
    }
    if (!saves.empty()) {
        itak_status st = save_ring_rows(pool, slot, *s, saves, save_elems);
        if (st != ITAK_OK) return st;
    }
    s->next_serial += 1;
    s->cp.live = true;
    s->cp.serial = s->next_serial;
    s->cp.max_round_tokens = max_round_tokens;
    s->cp.bases = s->appended;
    s->cp.ring_saves = std::move(saves);
    out->cache_id = s->cache_id;
    out->serial = s->cp.serial;
    out->max_round_tokens = max_round_tokens;
    // What the reference's snapshot of the evictable ring slots holds (cache.rs:678-697), as
    // the reference counts it (f32 rows of every windowed layer); the device sets rows aside
    // only on layers whose headroom the round outgrows, in the pool's element type.
    out->saved_bytes = windowed * max_round_tokens * 2 * pool->row * 4;
    ITAK_DIAG("checkpoint slot=%u serial=%llu max_round_tokens=%llu saved_bytes=%llu", slot,
              ULL(out->serial), ULL(max_round_tokens), ULL(out->saved_bytes));
    return ITAK_OK;
}

static itak_status live_data(itak_pool *pool, Slot &s, const itak_checkpoint *cp) {
    if (!cp) return invalid_argument(pool->err, "checkpoint is null");
    if (s.cp.live && s.cp.serial == cp->serial && cp->cache_id == s.cache_id) return ITAK_OK;
    return stale_checkpoint(pool->err, cp->serial);  // cache.rs:721-728
}

itak_status itak_kv_checkpoint_bases(itak_pool *pool, uint32_t slot, const itak_checkpoint *cp,
                                     uint64_t *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (!out || !cp) return invalid_argument(pool->err, "cp or out is null");
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    itak_status st = live_data(pool, *s, cp);
    if (st != ITAK_OK) return st;
    std::copy(s->cp.bases.begin(), s->cp.bases.end(), out);
    return ITAK_OK;
}

// A windowed layer can drop positions only while the rows written above the target have not
// wrapped onto rows the target's view still needs: with H the highest position ever written
// plus one, position x is overwritten once x + ring < H, and the view after the rewind starts
// at target - window, so H - target may be at most ring - window.
static itak_status check_ring_rewind(itak_pool *pool, const Slot &s, uint64_t target,
                                     const std::vector<RingSave> *saves = nullptr) {
    for (uint64_t li = 0; li < s.appended.size(); ++li) {
        const LayerInfo &L = pool->layers[li];
        if (!L.windowed || target >= s.appended[li]) continue;
        bool saved = false;  // a live checkpoint holds this layer's overwritten rows
        if (saves)
            for (const RingSave &rs : *saves) saved = saved || rs.layer == li;
        // A layer restored from a snapshot holds nothing older than the snapshot's first row.
        // The query appended next stands at `target` and sees down to target + 1 - window:
        // that must not reach under the first row. The lowest target that passes, first +
        // window - 1, is the resident session's rewind by one after a stored prefix covered
        // the whole prompt (crates/wgpu-compute/src/session.rs:5138-5143); the view at that
        // length has one row in it, the oldest, that was never written and reads as a fresh
        // ring's zeros, as after the reference's restore of fewer rows than the window.
        if (s.floor[li] > 0 && target + 1 < s.floor[li] + L.window)
            return rewind_range(pool->err, li, s.floor[li] + L.window - 1, s.appended[li], target);
        if (!saved && s.high[li] - target > L.ring - L.window)
            return set_error(pool->err, ITAK_CAPACITY_EXCEEDED, nullptr, li, s.high[li] - target,
                             L.ring - L.window, 0,
                             "dropping windowed layer %llu back to position %llu discards rows up to "
                             "%llu positions ahead of it, past the %llu rows of ring headroom; reset "
                             "the slot instead",
                             ULL(li), ULL(target), ULL(s.high[li] - target), ULL(L.ring - L.window));
    }
    return ITAK_OK;
}

// Drops positions >= target on every layer of the slot (the caller validated the range).
// Global layers truncate (cache.rs:788-791); windowed layers only move their length back: the
// dropped rows stay in the ring's headroom, out of every later query's window, until the
// positions are appended again.
static itak_status truncate_slots(itak_pool *pool, const uint32_t *slots, const uint64_t *targets,
                                  uint32_t count) {
    if ((pool->cfg.flags & ITAK_POOL_SCRUB_ON_TRUNCATE) && pool->global_layers) {
        for (uint32_t first = 0; first < count; first += kMaxBatchItems) {
            const uint32_t n = std::min<uint32_t>(kMaxBatchItems, count - first);
            ZeroBatch zb{};
            for (uint32_t i = 0; i < n; ++i) {
                const Slot &s = pool->slots[slots[first + i]];
                uint64_t max_len = 0;
                for (uint64_t li = 0; li < s.appended.size(); ++li)
                    if (!pool->layers[li].windowed) max_len = std::max(max_len, s.appended[li]);
                if (max_len <= targets[first + i]) continue;
                zb.item[zb.n++] = ZeroItem{slots[first + i], uint32_t(targets[first + i]),
                                           uint32_t(max_len), 0};
                zb.max_rows = std::max<uint32_t>(zb.max_rows, uint32_t(max_len - targets[first + i]));
            }
            itak_status st = scrub_rows(pool, zb);
            if (st != ITAK_OK) return st;
        }
    }
    for (uint32_t i = 0; i < count; ++i) {
        Slot &s = pool->slots[slots[i]];
        for (uint64_t li = 0; li < s.appended.size(); ++li) {
            s.appended[li] = std::min(s.appended[li], targets[i]);  // cache.rs:788-791,814
            // Scrubbed or not, a global layer's dropped rows are never read again.
            if (!pool->layers[li].windowed) s.high[li] = s.appended[li];
        }
    }
    return ITAK_OK;
}

itak_status itak_kv_rewind_to(itak_pool *pool, uint32_t slot, const itak_checkpoint *cp,
                              uint64_t target) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    itak_status st = live_data(pool, *s, cp);
    if (st != ITAK_OK) return st;
    // Validate every layer before touching any (cache.rs:772-783).
    for (uint64_t li = 0; li < s->appended.size(); ++li) {
        const uint64_t base = s->cp.bases[li];
        if (target < base || target > s->appended[li])
            return rewind_range(pool->err, li, base, s->appended[li], target);
    }
    st = check_ring_rewind(pool, *s, target, &s->cp.ring_saves);
    if (st != ITAK_OK) return st;
    ITAK_DIAG("rewind slot=%u serial=%llu target=%llu", slot, ULL(cp->serial), ULL(target));
    if (!s->cp.ring_saves.empty()) {
        // The rows the dropped positions overwrote come back from the checkpoint's copy
        // (cache.rs:792-812); what the ring then holds beyond `target` is what it held when
        // the checkpoint was taken.
        st = move_ring_rows(pool, slot, *s, s->cp.ring_saves, s->cp.bases.data(), target,
                            s->high.data(), true);
        if (st != ITAK_OK) return st;
        for (const RingSave &rs : s->cp.ring_saves)
            s->high[rs.layer] = std::max(target, std::min(rs.high0, s->high[rs.layer]));
    }
    return truncate_slots(pool, &slot, &target, 1);
}

itak_status itak_kv_release(itak_pool *pool, uint32_t slot, const itak_checkpoint *cp) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    itak_status st = live_data(pool, *s, cp);
    if (st != ITAK_OK) return st;
    s->cp.live = false;  // cache.rs:824-833
    s->cp.ring_saves.clear();
    ITAK_DIAG("release slot=%u serial=%llu", slot, ULL(cp->serial));
    return ITAK_OK;
}

itak_status itak_kv_truncate(itak_pool *pool, const uint32_t *slots, const uint64_t *new_lengths,
                             uint32_t count) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (count && (!slots || !new_lengths))
        return invalid_argument(pool->err, "slots or new_lengths is null");
    for (uint32_t i = 0; i < count; ++i) {
        Slot *s = find_slot(pool, slots[i]);
        if (!s) return invalid_argument(pool->err, "slot is not in use");
        if (s->cp.live) return checkpoint_busy(pool->err);
        for (uint64_t li = 0; li < s->appended.size(); ++li)
            if (new_lengths[i] > s->appended[li])
                return rewind_range(pool->err, li, 0, s->appended[li], new_lengths[i]);
        itak_status st = check_ring_rewind(pool, *s, new_lengths[i]);
        if (st != ITAK_OK) return st;
    }
    for (uint32_t i = 0; i < count; ++i)
        ITAK_DIAG("truncate slot=%u new_length=%llu", slots[i], ULL(new_lengths[i]));
    return truncate_slots(pool, slots, new_lengths, count);
}

itak_status itak_gqa_attention(itak_pool *pool, uint32_t slot, uint64_t layer, const float *q,
                               uint64_t q_len, uint64_t num_queries, uint64_t num_q_heads,
                               const uint64_t *query_positions, uint64_t positions_len,
                               float scale, float softcap, float *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    // attention.rs:115-146, in order.
    if (positions_len != num_queries)
        return shape_mismatch(pool->err, "query_positions", num_queries, positions_len);
    const uint64_t expected_q = num_queries * num_q_heads * pool->g.head_dim;
    if (q_len != expected_q) return shape_mismatch(pool->err, "q", expected_q, q_len);
    if (num_queries == 0) return ITAK_OK;
    if (num_q_heads == 0) return zero_dimension(pool->err, "num_q_heads");
    if (num_q_heads % pool->g.kv_heads != 0)
        return non_divisible(pool->err, num_q_heads, pool->g.kv_heads);
    if (!q || !out || !query_positions)
        return invalid_argument(pool->err, "q, out or query_positions is null");
    // The view holds positions oldest..appended; a query sees those at or below its own
    // position and inside its window (attention.rs:77-85,160-173).
    const uint64_t appended = s->appended[layer];
    const uint64_t oldest = first_visible(pool, *s, layer);
    const uint64_t window = pool->layers[layer].window;
    for (uint64_t i = 0; i < num_queries; ++i) {
        const uint64_t p = query_positions[i];
        const uint64_t newest_seen = std::min(p + 1, appended);  // exclusive
        const uint64_t oldest_seen =
            std::max(oldest, (window && p + 1 > window) ? p + 1 - window : 0);
        if (newest_seen <= oldest_seen) return no_visible_keys(pool->err, p);
    }
    if (std::isnan(scale)) scale = default_scale(pool->g.head_dim);

    bool consecutive = true;
    for (uint64_t i = 1; i < num_queries; ++i)
        consecutive = consecutive && query_positions[i] == query_positions[0] + i;
    const uint64_t q_bytes = align_up(q_len * sizeof(float), 256);
    const uint64_t pos_bytes = consecutive ? 0 : align_up(num_queries * sizeof(uint32_t), 256);
    itak_status st = ensure_stage(pool, 2 * q_bytes + pos_bytes);
    if (st != ITAK_OK) return st;
    float *qd = reinterpret_cast<float *>(pool->stage);
    uint32_t *pd = reinterpret_cast<uint32_t *>(pool->stage + q_bytes);
    float *od = reinterpret_cast<float *>(pool->stage + q_bytes + pos_bytes);
    std::vector<uint32_t> pos32;
    if (!consecutive) {
        pos32.resize(num_queries);
        for (uint64_t i = 0; i < num_queries; ++i)
            pos32[i] = uint32_t(std::min<uint64_t>(query_positions[i], 0xffffffffu));
    }
    const bool packed = 2 * q_bytes + pos_bytes <= kHostPacked;
    HostCall call;
    if (packed) {
        st = begin_host_call(pool, q_bytes + pos_bytes, q_len, call);
        if (st != ITAK_OK) return st;
        memcpy(call.in, q, q_len * 4);
        if (!consecutive) memcpy(call.in + q_bytes, pos32.data(), num_queries * 4);
        if (q_bytes + pos_bytes <= kHostByLaunch)
            HIP_TRY(pool, launch_stage_in(call.in_dev, qd, q_bytes + pos_bytes, pool->stream), "launch stage-in");
        else
            HIP_TRY(pool, hipMemcpyAsync(qd, call.in, q_bytes + pos_bytes, hipMemcpyHostToDevice, pool->stream), "upload q");
    } else {
        HIP_TRY(pool, hipMemcpyAsync(qd, q, q_len * 4, hipMemcpyHostToDevice, pool->stream), "upload q");
        if (!consecutive)
            HIP_TRY(pool, hipMemcpyAsync(pd, pos32.data(), num_queries * 4, hipMemcpyHostToDevice, pool->stream),
                    "upload query positions");
    }
    PlanInput pi{slot, uint32_t(num_queries),
                 uint32_t(std::min<uint64_t>(query_positions[0], 0xffffffffu - num_queries)),
                 uint32_t(appended), uint32_t(oldest)};
    st = run_attention(pool, layer, &pi, 1, qd, packed ? call.out_dev : od, consecutive ? nullptr : pd, num_q_heads, scale,
                       softcap);
    if (st != ITAK_OK) return st;
    if (packed) return finish_host_call(pool, call, out);
    HIP_TRY(pool, hipMemcpyAsync(out, od, q_len * 4, hipMemcpyDeviceToHost, pool->stream),
            "download attention output");
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after attention");
    return ITAK_OK;
}

// Append + attend for a validated plan. Decode and speculative blocks on f16 pools run as
// one launch that appends and attends (plus the split merge); other shapes append first.
static itak_status step_on_device(itak_pool *pool, uint64_t layer, const itak_batch_item *items,
                                  uint32_t item_count, const std::vector<PlanInput> &plan,
                                  const float *q_dev, const float *k_dev, const float *v_dev,
                                  float *out_dev, uint64_t num_q_heads, float scale,
                                  float softcap, const FoldedParams *folded = nullptr,
                                  bool no_alloc = false) {
    // Rows of zero-row items contribute nothing; q/k/v rows are numbered by walking the
    // items in order, so such items may simply be dropped.
    std::vector<PlanInput> &active = pool->active;
    active.clear();
    for (const PlanInput &p : plan)
        if (p.rows) active.push_back(p);
    uint32_t most_rows = 0;
    for (const PlanInput &p : active) most_rows = std::max(most_rows, p.rows);
    // Mid-size blocks on f16 pools: the block kernel in its one-tile form appends too.
    uint32_t most_blocks = 0;
    for (const PlanInput &p : active)
        most_blocks = std::max(most_blocks, (p.kv_len + 31) / 32 - p.kv_lo / 32);
    const bool splitk = takes_splitk_f16(pool, active.data(), uint32_t(active.size()), num_q_heads, nullptr);
    const bool any = !active.empty() &&
                     takes_splitk_any(pool, active.data(), uint32_t(active.size()), num_q_heads, q_dev, out_dev, nullptr);
    KernelChoice choice = choose_tiles(pool, layer, active.data(), uint32_t(active.size()), num_q_heads, softcap,
                                       folded && folded->prep_on, true, no_alloc);
    choice.in_place = shares_memory(pool, active.data(), uint32_t(active.size()), num_q_heads, out_dev, q_dev, k_dev, v_dev);
    // (With the queries as two halves the block kernel runs its two-tile form, which brings no
    // rows along: the append is a launch of its own.)
    const bool block_fuses =
        !splitk && !any && pool->elem_f16 && !active.empty() && !(pool->q_two_halves && pool->g.head_dim == 128) &&
        attn_prefill_f16_appends(pool->g, uint32_t(num_q_heads / pool->g.kv_heads), most_rows, most_blocks);
    const bool fuse =
        choice.tiles.sets ? choice.tiles.appends : splitk || block_fuses ||
        (!pool->elem_f16 && !active.empty() &&
         attn_splitk_f32_supports(pool->g, uint32_t(num_q_heads / pool->g.kv_heads), most_rows)) ||
        (any && aligned16(k_dev) && aligned16(v_dev) &&
         attn_splitk_any_appends(pool->g, pool->elem_f16, uint32_t(num_q_heads / pool->g.kv_heads), most_rows));
    // The allocation-free form plans first and refuses, before anything changes, a step whose
    // launches need more workspace than the static array has.
    struct NoAllocScope {
        itak_pool *pool;
        bool on;
        ~NoAllocScope() { if (on) pool->no_alloc_call = false; }
    } scope{pool, no_alloc};
    if (no_alloc) {
        WorkspaceNeed need;
        itak_status st = run_attention(pool, layer, active.data(), uint32_t(active.size()), q_dev, out_dev,
                                       nullptr, num_q_heads, scale, softcap, nullptr, nullptr, folded,
                                       &need, &choice);
        if (st != ITAK_OK) return st;
        const uint64_t partial_bytes = need.partial_floats * sizeof(float);
        const uint64_t exchange_bytes = need.exchange_words * 8;
        if (partial_bytes > kScratchBytes - kScratchExchangeBytes)
            return set_error(pool->err, ITAK_CAPACITY_EXCEEDED, "split workspace", layer, partial_bytes,
                             kScratchBytes - kScratchExchangeBytes, 0,
                             "the step's split partials need %llu bytes of workspace and the "
                             "allocation-free entry point holds %llu: use fewer slots or rows per "
                             "step, or itak_attention_step_device",
                             ULL(partial_bytes), ULL(kScratchBytes - kScratchExchangeBytes));
        if (exchange_bytes > kScratchExchangeBytes)
            return set_error(pool->err, ITAK_CAPACITY_EXCEEDED, "split workspace", layer, exchange_bytes,
                             kScratchExchangeBytes, 0,
                             "the step's split exchange needs %llu bytes of workspace and the "
                             "allocation-free entry point holds %llu: use fewer slots or rows per "
                             "step, or itak_attention_step_device",
                             ULL(exchange_bytes), ULL(kScratchExchangeBytes));
        pool->no_alloc_call = true;
        if (need.exchange_words) pool->scratch_exchange_used = true;
    }
    if (fuse) {
        for (uint32_t i = 0; i < item_count; ++i)
            advance(pool->slots[items[i].slot], layer, items[i].rows);
        return run_attention(pool, layer, active.data(), uint32_t(active.size()), q_dev, out_dev,
                             nullptr, num_q_heads, scale, softcap, k_dev, v_dev, folded, nullptr, &choice);
    }
    itak_status st = run_append(pool, layer, items, item_count, k_dev, v_dev);
    if (st != ITAK_OK) return st;
    return run_attention(pool, layer, active.data(), uint32_t(active.size()), q_dev, out_dev,
                         nullptr, num_q_heads, scale, softcap, nullptr, nullptr, folded, nullptr, &choice);
}

// Validates one batched step and returns the per-item plan (positions before the append).
static itak_status plan_step(itak_pool *pool, uint64_t layer, const itak_batch_item *items,
                             uint32_t item_count, uint64_t num_q_heads,
                             std::vector<PlanInput> &plan) {
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (num_q_heads == 0) return zero_dimension(pool->err, "num_q_heads");
    if (num_q_heads % pool->g.kv_heads != 0)
        return non_divisible(pool->err, num_q_heads, pool->g.kv_heads);
    std::vector<uint64_t> &named = pool->named;
    named.resize(pool->slots.size(), 0);
    const uint64_t number = ++pool->step_number;
    plan.clear();
    for (uint32_t i = 0; i < item_count; ++i) {
        Slot *s = find_slot(pool, items[i].slot);
        if (!s) return invalid_argument(pool->err, "slot is not in use");
        if (named[items[i].slot] == number) return invalid_argument(pool->err, "slot listed twice in one step");
        named[items[i].slot] = number;
        uint64_t ok = 0;
        itak_status st = check_append_rows(pool, *s, layer, items[i].rows, &ok);
        if (st != ITAK_OK) return st;
        st = check_block_rows(pool, layer, items[i].rows);
        if (st != ITAK_OK) return st;
        const uint64_t base = s->appended[layer];
        // The block's first row still sees its whole window: the rows below the view of the
        // block's end are kept by the ring's headroom.
        const uint64_t window = pool->layers[layer].window;
        const uint64_t lo = (window && base + 1 > window) ? base + 1 - window : 0;
        plan.push_back(PlanInput{items[i].slot, items[i].rows, uint32_t(base),
                                 uint32_t(base + items[i].rows), uint32_t(lo)});
    }
    return ITAK_OK;
}

itak_status itak_attention_step_device(itak_pool *pool, uint64_t layer,
                                       const itak_batch_item *items, uint32_t item_count,
                                       const float *q_dev, const float *k_dev, const float *v_dev,
                                       float *out_dev, uint64_t num_q_heads, float scale,
                                       float softcap) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (item_count == 0) return ITAK_OK;
    if (!items || !q_dev || !k_dev || !v_dev || !out_dev)
        return invalid_argument(pool->err, "items or a device tensor is null");
    std::vector<PlanInput> &plan = pool->plan;
    itak_status st = plan_step(pool, layer, items, item_count, num_q_heads, plan);
    if (st != ITAK_OK) return st;
    if (std::isnan(scale)) scale = default_scale(pool->g.head_dim);
    return step_on_device(pool, layer, items, item_count, plan, q_dev, k_dev, v_dev, out_dev,
                          num_q_heads, scale, softcap);
}

itak_status itak_attention_step_device_noalloc(itak_pool *pool, uint64_t layer,
                                               const itak_batch_item *items, uint32_t item_count,
                                               const float *q_dev, const float *k_dev,
                                               const float *v_dev, float *out_dev,
                                               uint64_t num_q_heads, float scale, float softcap) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (item_count == 0) return ITAK_OK;
    if (!items || !q_dev || !k_dev || !v_dev || !out_dev)
        return invalid_argument(pool->err, "items or a device tensor is null");
    std::vector<PlanInput> &plan = pool->plan;
    itak_status st = plan_step(pool, layer, items, item_count, num_q_heads, plan);
    if (st != ITAK_OK) return st;
    if (std::isnan(scale)) scale = default_scale(pool->g.head_dim);
    bool capturing = false;
    HIP_TRY(pool, scratch_guard_enter(pool->cfg.device, pool->stream, &capturing),
            "order the step behind the static workspace's last user");
    st = step_on_device(pool, layer, items, item_count, plan, q_dev, k_dev, v_dev, out_dev,
                        num_q_heads, scale, softcap, nullptr, true);
    if (!capturing)
        HIP_TRY(pool, scratch_guard_leave(pool->cfg.device, pool->stream),
                "mark the static workspace's last user");
    return st;
}

itak_status itak_attention_prep_step_device(itak_pool *pool, uint64_t layer,
                                            const itak_batch_item *items, uint32_t item_count,
                                            const float *q_dev, const float *k_dev,
                                            const float *v_dev, const float *gate_dev,
                                            float *out_dev, uint64_t num_q_heads, float scale,
                                            float softcap, const itak_prep_params *prep) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (item_count == 0) return ITAK_OK;
    if (!items || !q_dev || !k_dev || !v_dev || !out_dev || !prep)
        return invalid_argument(pool->err, "items, a device tensor or prep is null");
    const uint32_t D = pool->g.head_dim;
    // torch-math's refusals (norm.rs:32-38, rope_interleaved.rs:72-99), by name.
    if ((prep->q_norm_weight || prep->k_norm_weight) && !(std::isfinite(prep->eps) && prep->eps > 0.0f))
        return set_error(pool->err, ITAK_STEP_FAILED, "rms_norm", 0, 0, 0, 0,
                         "rms_norm: eps must be finite and > 0");
    const bool rotate = prep->rope_base != 0.0f;
    const uint32_t rotary = prep->rotary_dim ? prep->rotary_dim : D;
    if (rotate) {
        if (D < 2 || D % 2 != 0)
            return set_error(pool->err, ITAK_STEP_FAILED, "attention", 0, 0, 0, 0,
                             "rope: head_dim must be even and >= 2");
        if (rotary < 2 || rotary % 2 != 0 || rotary > D)
            return set_error(pool->err, ITAK_STEP_FAILED, "attention", 0, 0, 0, 0,
                             "rope: rotary_dim must be even, >= 2, and <= head_dim");
        if (!std::isfinite(prep->rope_base) || prep->rope_base <= 1.0f)
            return set_error(pool->err, ITAK_STEP_FAILED, "attention", 0, 0, 0, 0,
                             "rope: base must be finite and > 1");
    } else if (D % 2 != 0) {
        return unsupported(pool->err, "attention preparation needs an even head_dim");
    }
    std::vector<PlanInput> &plan = pool->plan;
    itak_status st = plan_step(pool, layer, items, item_count, num_q_heads, plan);
    if (st != ITAK_OK) return st;
    uint64_t total_rows = 0;
    for (const PlanInput &p : plan) total_rows += p.rows;
    if (total_rows == 0) return ITAK_OK;
    const uint64_t q_width = num_q_heads * D, k_width = pool->row;
    if (std::isnan(scale)) scale = default_scale(D);
    // Steps the split-K kernel takes (decode, speculative blocks: up to 64 query vectors per KV
    // head) have Q and the new K rows prepared by that kernel and the gate applied by the
    // kernel that writes the output: no launch but the step's own two.
    std::vector<PlanInput> &active = pool->active;  // step_on_device fills it again, with the same
    active.clear();
    for (const PlanInput &p : plan)
        if (p.rows) active.push_back(p);
    const bool splitk = takes_splitk_f16(pool, active.data(), uint32_t(active.size()), num_q_heads,
                                         nullptr);
    const bool interleaved = prep->rope_interleaved != 0;
    const bool folds = splitk && !pool->prep_by_launch && (!rotate || interleaved || rotary % 8 == 0);
    FoldedParams folded{};
    folded.gate = gate_dev;
    if (folds) {
        folded.prep_on = 1;
        folded.prep_interleaved = interleaved ? 1 : 0;
        folded.prep_rot = rotate ? rotary : 0;
        folded.prep_eps = prep->eps;
        folded.prep_q_weight = prep->q_norm_weight;
        folded.prep_k_weight = prep->k_norm_weight;
        // Pair i turns at position * base^(-2i/rot) = position * 2^(i * step).
        folded.prep_freq = rotate ? rope_freq_table(pool, prep->rope_base, rotary) : nullptr;
        folded.prep_freq_step = rotate ? -2.0 * std::log2(double(prep->rope_base)) / double(rotary) : 0.0;
        return step_on_device(pool, layer, items, item_count, plan, q_dev, k_dev, v_dev, out_dev,
                              num_q_heads, scale, softcap, &folded);
    }
    st = ensure_prep(pool, total_rows * (q_width + k_width));
    if (st != ITAK_OK) return st;
    float *q_prep = pool->prep, *k_prep = pool->prep + total_rows * q_width;
    uint32_t row = 0;
    for (uint32_t first = 0; first < item_count; first += kMaxBatchItems) {
        const uint32_t count = std::min<uint32_t>(kMaxBatchItems, item_count - first);
        PrepArgs a{};
        a.q_in = q_dev + uint64_t(row) * q_width;
        a.k_in = k_dev + uint64_t(row) * k_width;
        a.q_out = q_prep + uint64_t(row) * q_width;
        a.k_out = k_prep + uint64_t(row) * k_width;
        a.q_weight = prep->q_norm_weight;
        a.k_weight = prep->k_norm_weight;
        a.eps = prep->eps;
        a.rope_base = rotate ? prep->rope_base : 0.0f;
        a.rope_freq = rotate ? rope_freq_table(pool, prep->rope_base, rotary) : nullptr;
        a.interleaved = interleaved ? 1 : 0;
        a.rotary_dim = rotary;
        a.head_dim = D;
        a.q_heads = uint32_t(num_q_heads);
        a.kv_heads = pool->g.kv_heads;
        a.n = count;
        uint32_t chunk_rows = 0;
        for (uint32_t i = 0; i < count; ++i) {
            a.row0[i] = chunk_rows;
            a.pos0[i] = plan[first + i].pos0;
            chunk_rows += plan[first + i].rows;
        }
        a.total_rows = chunk_rows;
        HIP_TRY(pool, launch_attn_prep(a, pool->stream), "launch attention preparation");
        row += chunk_rows;
    }
    return step_on_device(pool, layer, items, item_count, plan, q_prep, k_prep, v_dev, out_dev,
                          num_q_heads, scale, softcap, &folded);
}

itak_status itak_attention_device(itak_pool *pool, uint64_t layer, const itak_batch_item *items,
                                  uint32_t item_count, const float *q_dev, float *out_dev,
                                  uint64_t num_q_heads, float scale, float softcap) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (item_count == 0) return ITAK_OK;
    if (!items || !q_dev || !out_dev)
        return invalid_argument(pool->err, "items or a device tensor is null");
    if (layer >= pool->cfg.layer_count) return invalid_layer(pool->err, layer, pool->cfg.layer_count);
    if (num_q_heads == 0) return zero_dimension(pool->err, "num_q_heads");
    if (num_q_heads % pool->g.kv_heads != 0)
        return non_divisible(pool->err, num_q_heads, pool->g.kv_heads);
    std::vector<PlanInput> plan;
    for (uint32_t i = 0; i < item_count; ++i) {
        Slot *s = find_slot(pool, items[i].slot);
        if (!s) return invalid_argument(pool->err, "slot is not in use");
        const uint64_t len = s->appended[layer];
        if (items[i].rows == 0) continue;
        if (len == 0) return no_visible_keys(pool->err, 0);
        if (items[i].rows > len)
            return shape_mismatch(pool->err, "query rows", len, items[i].rows);
        // The newest `rows` positions query the view as it stands: nothing older than the
        // view's first row is promised to be in the ring. A query that stands before that row
        // (more rows than a windowed layer's window) sees none of the view: the reference's
        // refusal for its position (attention.rs:160-173), the lowest such query first.
        const uint64_t first = first_visible(pool, *s, layer);
        if (len - items[i].rows < first) return no_visible_keys(pool->err, len - items[i].rows);
        plan.push_back(PlanInput{items[i].slot, items[i].rows, uint32_t(len - items[i].rows),
                                 uint32_t(len), uint32_t(first)});
    }
    if (std::isnan(scale)) scale = default_scale(pool->g.head_dim);
    return run_attention(pool, layer, plan.data(), uint32_t(plan.size()), q_dev, out_dev, nullptr,
                         num_q_heads, scale, softcap);
}

itak_status itak_compute_attention(itak_pool *pool, uint32_t slot, uint64_t layer, const float *q,
                                   uint64_t q_len, const float *k, uint64_t k_len, const float *v,
                                   uint64_t v_len, uint64_t num_q_heads, uint64_t cache_position,
                                   float softcap, float rope_freq_base_swa, float *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    const char *step = "attention";
    // cpu.rs:529-556: whole rows, matching K/V row counts.
    const uint64_t q_width = num_q_heads * pool->g.head_dim;
    if (q_width == 0 || q_len % q_width != 0)
        return set_error(pool->err, ITAK_STEP_FAILED, step, q_len, q_width, 0, 0,
                         "query projection holds %llu elements, not a whole number of "
                         "%llu-wide rows",
                         ULL(q_len), ULL(q_width));
    const uint64_t rows = q_len / q_width;
    if (k_len != rows * pool->row || v_len != rows * pool->row)
        return set_error(pool->err, ITAK_STEP_FAILED, step, k_len, v_len, rows * pool->row, 0,
                         "key/value projections hold %llu/%llu elements for %llu rows, expected "
                         "%llu/%llu",
                         ULL(k_len), ULL(v_len), ULL(rows), ULL(rows * pool->row),
                         ULL(rows * pool->row));
    if (layer >= pool->cfg.layer_count) {
        invalid_layer(pool->err, layer, pool->cfg.layer_count);
        pool->err.info.code = ITAK_STEP_FAILED;  // forwarded as StepFailed text (cpu.rs:565-568)
        return ITAK_STEP_FAILED;
    }
    s->built = true;  // KvState::build on first use (cpu.rs:560-564)
    const uint64_t appended = s->appended[layer];
    if (appended != cache_position)  // cpu.rs:569-581
        return set_error(pool->err, ITAK_STEP_FAILED, step, layer, appended, cache_position, 0,
                         "KV state for layer %llu is at position %llu but the sequence cache is "
                         "at position %llu: the two disagree, so attending would read the wrong "
                         "history. Pair one Cache with one compute slot per sequence, or reset "
                         "the slot when a sequence is abandoned (a forward that failed midway "
                         "leaves the KV state ahead of the cache and also needs a reset)",
                         ULL(layer), ULL(appended), ULL(cache_position));
    if (rows == 0) return ITAK_OK;
    if (num_q_heads % pool->g.kv_heads != 0) {
        non_divisible(pool->err, num_q_heads, pool->g.kv_heads);
        pool->err.info.code = ITAK_STEP_FAILED;
        return ITAK_STEP_FAILED;
    }
    if (!q || !k || !v || !out) return invalid_argument(pool->err, "q, k, v or out is null");
    // Sliding-window layers rotate Q and K (cpu.rs:594-622); torch_math::rope_interleaved's
    // refusals (rope_interleaved.rs:72-99) surface under the attention step.
    const bool rotate = pool->layers[layer].windowed;
    if (rotate) {
        if (pool->g.head_dim < 2 || pool->g.head_dim % 2 != 0)
            return set_error(pool->err, ITAK_STEP_FAILED, step, 0, 0, 0, 0,
                             "rope: head_dim must be even and >= 2");
        if (!std::isfinite(rope_freq_base_swa) || rope_freq_base_swa <= 1.0f)
            return set_error(pool->err, ITAK_STEP_FAILED, step, 0, 0, 0, 0,
                             "rope: base must be finite and > 1");
    }

    // Row-at-a-time appends stop at the first refusal (cpu.rs:623-631): rows before it are
    // in the cache when the call fails, exactly as in the reference.
    uint64_t ok_rows = rows;
    itak_status refusal = check_append_rows(pool, *s, layer, rows, &ok_rows);
    ErrorState saved = pool->err;

    const uint64_t q_bytes = align_up(q_len * sizeof(float), 256);
    const uint64_t kv_bytes = align_up(k_len * sizeof(float), 256);
    itak_status st = ensure_stage(pool, 2 * q_bytes + 2 * kv_bytes);
    if (st != ITAK_OK) return st;
    float *qd = reinterpret_cast<float *>(pool->stage);
    float *kd = reinterpret_cast<float *>(pool->stage + q_bytes);
    float *vd = reinterpret_cast<float *>(pool->stage + q_bytes + kv_bytes);
    float *od = reinterpret_cast<float *>(pool->stage + q_bytes + 2 * kv_bytes);
    const float *q_src = qd, *k_src = kd, *v_src = vd;  // where the first kernel that reads them finds them
    const uint64_t in_bytes = q_bytes + 2 * kv_bytes;
    const bool packed = in_bytes + q_bytes <= kHostPacked;
    HostCall call;
    if (packed) {
        st = begin_host_call(pool, in_bytes, q_len, call);
        if (st != ITAK_OK) return st;
        memcpy(call.in, q, q_len * 4);
        memcpy(call.in + q_bytes, k, k_len * 4);
        memcpy(call.in + q_bytes + kv_bytes, v, v_len * 4);
        // Where everything is read once or nearly so, the kernels read it in pinned memory and the
        // launch that would fetch it goes away: the rotation reads Q and K once, the workgroups that
        // append the new rows read those, and every split of a KV head's keys its queries (four key
        // blocks or more a split; 64 KB over the link is what the launch costs).
        const uint64_t key_blocks = (appended + rows + 31) / 32;
        const uint64_t q_reads = rotate ? 1 : std::max<uint64_t>((key_blocks + 3) / 4, 1);
        const bool in_place = q_len * 4 * q_reads + 2 * k_len * 4 <= (64u << 10);
        if (in_place) {
            q_src = reinterpret_cast<const float *>(call.in_dev);
            k_src = reinterpret_cast<const float *>(call.in_dev + q_bytes);
            v_src = reinterpret_cast<const float *>(call.in_dev + q_bytes + kv_bytes);
        } else if (in_bytes <= kHostByLaunch) {
            HIP_TRY(pool, launch_stage_in(call.in_dev, qd, in_bytes, pool->stream), "launch stage-in");
        } else {
            HIP_TRY(pool, hipMemcpyAsync(qd, call.in, in_bytes, hipMemcpyHostToDevice, pool->stream),
                    "upload q, k, v");
        }
    } else {
        HIP_TRY(pool, hipMemcpyAsync(kd, k, k_len * 4, hipMemcpyHostToDevice, pool->stream), "upload k");
        HIP_TRY(pool, hipMemcpyAsync(vd, v, v_len * 4, hipMemcpyHostToDevice, pool->stream), "upload v");
        HIP_TRY(pool, hipMemcpyAsync(qd, q, q_len * 4, hipMemcpyHostToDevice, pool->stream), "upload q");
    }
    // The reference appends and attends row by row (cpu.rs:586-646). Here a block is appended
    // whole and attended under the causal mask, which is the same thing on a global layer; on
    // a windowed layer a block may be as long as the ring's headroom, so longer inputs go in
    // several blocks.
    const LayerInfo &L = pool->layers[layer];
    const uint64_t block_cap = L.windowed ? L.ring - L.window : std::max<uint64_t>(rows, 1);
    // The rotation of a sliding-window layer (row i at position appended + i): by the preparation
    // launch, whose f64 angles, sines and cosines are the
    // reference's (rope_interleaved.rs:103-114), so that the K rows this call stores are the
    // reference's rounded once. (The split-K kernel can rotate inside its own launch, with the
    // hardware's sine and cosine, within one f16 step of that; the device-resident step uses it,
    // where a launch counts. Here the call already copies its rows in and its output out.)
    auto rotate_block = [&](uint64_t done, uint64_t n, bool with_q) -> itak_status {
        PrepArgs a{};
        a.q_in = q_src + done * q_width;
        a.q_out = qd + done * q_width;
        a.k_in = k_src + done * pool->row;
        a.k_out = kd + done * pool->row;
        a.rope_base = rope_freq_base_swa;
        a.rope_freq = rope_freq_table(pool, rope_freq_base_swa, pool->g.head_dim);
        a.interleaved = 1;
        a.rotary_dim = pool->g.head_dim;
        a.head_dim = pool->g.head_dim;
        a.q_heads = with_q ? uint32_t(num_q_heads) : 0;
        a.kv_heads = pool->g.kv_heads;
        a.total_rows = uint32_t(n);
        a.n = 1;
        a.row0[0] = 0;
        a.pos0[0] = uint32_t(appended + done);
        HIP_TRY(pool, launch_attn_prep(a, pool->stream), "launch rope");
        return ITAK_OK;
    };
    if (refusal != ITAK_OK) {
        for (uint64_t done = 0; done < ok_rows; done += block_cap) {
            const uint64_t n = std::min(block_cap, ok_rows - done);
            if (rotate && (st = rotate_block(done, n, false)) != ITAK_OK) return st;
            itak_batch_item item{slot, uint32_t(n)};
            st = run_append(pool, layer, &item, 1, (rotate ? kd : k_src) + done * pool->row, v_src + done * pool->row);
            if (st != ITAK_OK) return st;
        }
        HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after append");
        pool->turns.drained();
        pool->err = saved;
        pool->err.info.code = ITAK_STEP_FAILED;
        return ITAK_STEP_FAILED;
    }
    float *out_dev = packed ? call.out_dev : od;
    for (uint64_t done = 0; done < rows; done += block_cap) {
        const uint64_t n = std::min(block_cap, rows - done);
        itak_batch_item item{slot, uint32_t(n)};
        const uint64_t base = appended + done;
        const uint64_t lo = (L.window && base + 1 > L.window) ? base + 1 - L.window : 0;
        std::vector<PlanInput> plan{
            PlanInput{slot, uint32_t(n), uint32_t(base), uint32_t(base + n), uint32_t(lo)}};
        if (rotate && (st = rotate_block(done, n, true)) != ITAK_OK) return st;
        st = step_on_device(pool, layer, &item, 1, plan, (rotate ? qd : q_src) + done * q_width,
                            (rotate ? kd : k_src) + done * pool->row, v_src + done * pool->row, out_dev + done * q_width, num_q_heads,
                            default_scale(pool->g.head_dim),  // AttentionParams::new(), cpu.rs:584
                            softcap, nullptr);
        if (st != ITAK_OK) return st;
    }
    if (packed) return finish_host_call(pool, call, out);
    HIP_TRY(pool, hipMemcpyAsync(out, od, q_len * 4, hipMemcpyDeviceToHost, pool->stream),
            "download attention output");
    HIP_TRY(pool, hipStreamSynchronize(pool->stream), "synchronize after attention");
    return ITAK_OK;
}

static itak_status no_kv_state(itak_pool *pool, const char *step, const char *detail) {
    return set_error(pool->err, ITAK_STEP_FAILED, step, 0, 0, 0, 0, "%s", detail);
}

static itak_status as_step_failed(itak_pool *pool, itak_status st) {
    if (st == ITAK_OK) return st;
    pool->err.info.code = ITAK_STEP_FAILED;  // map_err(step_failed(...)) in cpu.rs:292-294
    return ITAK_STEP_FAILED;
}

itak_status itak_compute_cache_checkpoint(itak_pool *pool, uint32_t slot,
                                          uint64_t max_round_tokens, itak_checkpoint *out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!s->built)  // cpu.rs:284-290
        return no_kv_state(pool, "cache_checkpoint",
                           "no KV state exists yet: a speculative round checkpoints after a first "
                           "forward has built the cache (the spec's prefill), not before");
    return as_step_failed(pool, itak_kv_checkpoint(pool, slot, max_round_tokens, out));
}

itak_status itak_compute_cache_rewind(itak_pool *pool, uint32_t slot, const itak_checkpoint *cp,
                                      uint64_t target) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!s->built)  // cpu.rs:311-317
        return no_kv_state(pool, "cache_rewind",
                           "no KV state exists: the sequence was reset after the checkpoint was "
                           "taken");
    return as_step_failed(pool, itak_kv_rewind_to(pool, slot, cp, target));
}

itak_status itak_compute_cache_release(itak_pool *pool, uint32_t slot, const itak_checkpoint *cp) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    Slot *s = find_slot(pool, slot);
    if (!s) return invalid_argument(pool->err, "slot is not in use");
    if (!s->built)  // cpu.rs:327-333
        return no_kv_state(pool, "cache_release",
                           "no KV state exists: the sequence was reset after the checkpoint was "
                           "taken");
    return as_step_failed(pool, itak_kv_release(pool, slot, cp));
}

itak_status itak_convert_f32_to_f16_device(itak_pool *pool, const float *src_dev,
                                           uint16_t *dst_dev, uint64_t count) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (count && (!src_dev || !dst_dev)) return invalid_argument(pool->err, "src or dst is null");
    HIP_TRY(pool, launch_convert_f16(src_dev, dst_dev, count, pool->stream), "launch conversion");
    return ITAK_OK;
}

itak_status itak_probe_copy_device(itak_pool *pool, const void *src_dev, void *dst_dev,
                                   uint64_t bytes) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (bytes && (!src_dev || !dst_dev)) return invalid_argument(pool->err, "src or dst is null");
    if (bytes % 16 != 0) return invalid_argument(pool->err, "bytes is not a multiple of 16");
    HIP_TRY(pool, launch_probe_copy(src_dev, dst_dev, bytes, pool->stream), "launch probe copy");
    return ITAK_OK;
}

itak_status itak_probe_read_device(itak_pool *pool, const void *src_dev, uint64_t bytes) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (bytes && !src_dev) return invalid_argument(pool->err, "src is null");
    if (bytes % 16 != 0) return invalid_argument(pool->err, "bytes is not a multiple of 16");
    HIP_TRY(pool, launch_probe_read(src_dev, bytes, pool->stream), "launch probe read");
    return ITAK_OK;
}

void itak_set_debug_enabled(int32_t enabled) {
    g_debug_enabled.store(enabled != 0, std::memory_order_relaxed);
}
int32_t itak_debug_enabled(void) { return diag_enabled() ? 1 : 0; }

itak_status itak_probe_empty_launch(itak_pool *pool) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    HIP_TRY(pool, launch_probe_empty(pool->stream), "launch empty probe");
    return ITAK_OK;
}

itak_status itak_probe_mfma(itak_pool *pool, uint32_t random_operands, uint32_t trips,
                            uint64_t *clocks_dev, uint64_t *flops_out) {
    if (!pool) return ITAK_INVALID_ARGUMENT;
    if (trips == 0 || trips > (1u << 22)) return invalid_argument(pool->err, "trips is not in 1 ..= 2^22");
    uint32_t workgroups = 0;
    HIP_TRY(pool,
            launch_probe_mfma(random_operands != 0, trips,
                              reinterpret_cast<unsigned long long *>(clocks_dev), &workgroups, pool->stream),
            "launch MFMA probe");
    // 4 wavefronts a workgroup, 32 products a trip, 16 x 16 x 32 multiply-adds a product.
    if (flops_out) *flops_out = uint64_t(workgroups) * 4u * uint64_t(trips) * 32u * 16384u;
    return ITAK_OK;
}

}  // extern "C"
