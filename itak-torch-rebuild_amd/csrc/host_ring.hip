// Host code: see host_ring.h.
#include "host_ring.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <thread>

#include "itkv.h"

namespace itak {

hipError_t HostRing::open(uint64_t slots) {
    for (uint64_t i = 0; i < std::min<uint64_t>(slots, kRingSlots); ++i) {
        hipError_t e = hipSuccess;
        if (!moved[i]) e = hipEventCreateWithFlags(&moved[i], hipEventDisableTiming);
        if (e == hipSuccess && !slot[i])
            e = hipHostMalloc(reinterpret_cast<void **>(&slot[i]), kRingChunk, hipHostMallocDefault);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

void HostRing::close() {
    for (unsigned char *&p : slot) {
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
    for (hipEvent_t &e : moved) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

namespace {

struct Chunk {
    const unsigned char *src;
    unsigned char *dst;
    uint64_t bytes;
};

// What the threads of one transfer share. Chunk c uses slot c % kRingSlots; thread w of `workers`
// has the chunks w, w + workers, ..
struct Transfer {
    std::atomic<uint64_t> enqueued{0};              // chunks whose copy command and event are on the stream
    std::atomic<uint64_t> host_done[kRingSlots];    // per slot: 1 + the last chunk the host has filled / emptied
    std::atomic<int> error{0};
    Transfer() {
        for (auto &x : host_done) x.store(0, std::memory_order_relaxed);
    }
    // False when another thread has failed meanwhile.
    template <class F>
    bool wait(F ready) {
        for (uint32_t looks = 0; !ready(); ++looks) {
            if (error.load(std::memory_order_relaxed)) return false;
            if (looks > 64) std::this_thread::yield();
        }
        return error.load(std::memory_order_relaxed) == 0;
    }
    void fail(hipError_t e) {
        int none = 0;
        error.compare_exchange_strong(none, int(e));
    }
};

// Runs work(w, workers) on helper threads beside drive() on this one.
template <class Work, class Drive>
hipError_t run_transfer(Transfer &t, uint64_t chunks, Work work, Drive drive) {
    int device = 0;
    if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
    const uint64_t want = std::min<uint64_t>({uint64_t(host_threads()), chunks, uint64_t(kRingSlots)});
    std::vector<std::thread> helpers;
    std::atomic<uint64_t> workers{0};  // known once every helper that can be had is there
    for (uint64_t i = 0; i < want; ++i) {
        try {
            helpers.emplace_back([&, i] {
                if (hipError_t e = hipSetDevice(device); e != hipSuccess) return t.fail(e);
                while (workers.load() == 0) std::this_thread::yield();
                work(i, workers.load());
            });
        } catch (...) {
            break;
        }
    }
    if (helpers.empty()) return hipErrorOutOfMemory;
    workers.store(helpers.size());
    drive();
    for (std::thread &h : helpers) h.join();
    return hipError_t(t.error.load());
}

}  // namespace

hipError_t ring_upload(HostRing &ring, const std::vector<RingSpan> &spans, hipStream_t stream,
                       const std::function<hipError_t(uint64_t)> &after) {
    std::vector<Chunk> chunks;
    for (const RingSpan &s : spans)
        for (uint64_t at = 0; at < s.bytes; at += kRingChunk)
            chunks.push_back(Chunk{static_cast<const unsigned char *>(s.src) + at, static_cast<unsigned char *>(s.dst) + at,
                                   std::min(kRingChunk, s.bytes - at)});
    if (chunks.empty()) return hipSuccess;
    if (hipError_t e = ring.open(chunks.size()); e != hipSuccess) return e;
    Transfer t;
    auto fill = [&](uint64_t first, uint64_t step) {
        for (uint64_t c = first; c < chunks.size(); c += step) {
            const uint32_t slot = c % kRingSlots;
            if (c >= kRingSlots) {
                if (!t.wait([&] { return t.enqueued.load(std::memory_order_acquire) > c - kRingSlots; })) return;
                if (hipError_t e = hipEventSynchronize(ring.moved[slot]); e != hipSuccess) return t.fail(e);
            }
            memcpy(ring.slot[slot], chunks[c].src, chunks[c].bytes);
            t.host_done[slot].store(c + 1, std::memory_order_release);
        }
    };
    auto drive = [&] {
        uint64_t sent = 0;
        for (uint64_t c = 0; c < chunks.size(); ++c) {
            const uint32_t slot = c % kRingSlots;
            if (!t.wait([&] { return t.host_done[slot].load(std::memory_order_acquire) == c + 1; })) return;
            hipError_t e = hipMemcpyAsync(chunks[c].dst, ring.slot[slot], chunks[c].bytes,
                                          hipMemcpyHostToDevice, stream);
            if (e == hipSuccess) e = hipEventRecord(ring.moved[slot], stream);
            sent += chunks[c].bytes;
            if (e == hipSuccess) t.enqueued.store(c + 1, std::memory_order_release);
            if (e == hipSuccess && after) e = after(sent);
            if (e != hipSuccess) return t.fail(e);
        }
    };
    if (chunks.size() == 1) {  // nothing to overlap
        fill(0, 1);
        drive();
        return hipError_t(t.error.load());
    }
    return run_transfer(t, chunks.size(), fill, drive);
}

hipError_t ring_download(HostRing &ring, void *out, uint64_t bytes, hipStream_t stream,
                         const std::function<hipError_t(uint64_t, uint64_t, const void **)> &source) {
    if (bytes == 0) return hipSuccess;
    const uint64_t chunks = (bytes + kRingChunk - 1) / kRingChunk;
    if (hipError_t e = ring.open(chunks); e != hipSuccess) return e;
    unsigned char *to = static_cast<unsigned char *>(out);
    auto size_of = [&](uint64_t c) { return std::min(kRingChunk, bytes - c * kRingChunk); };
    Transfer t;
    auto drive = [&] {
        for (uint64_t c = 0; c < chunks; ++c) {
            const uint32_t slot = c % kRingSlots;
            if (c >= kRingSlots &&
                !t.wait([&] { return t.host_done[slot].load(std::memory_order_acquire) == c - kRingSlots + 1; }))
                return;
            const void *from = nullptr;
            hipError_t e = source(c * kRingChunk, size_of(c), &from);
            if (e == hipSuccess)
                e = hipMemcpyAsync(ring.slot[slot], from, size_of(c), hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(ring.moved[slot], stream);
            if (e != hipSuccess) return t.fail(e);
            t.enqueued.store(c + 1, std::memory_order_release);
        }
    };
    auto empty = [&](uint64_t first, uint64_t step) {
        for (uint64_t c = first; c < chunks; c += step) {
            const uint32_t slot = c % kRingSlots;
            if (!t.wait([&] { return t.enqueued.load(std::memory_order_acquire) > c; })) return;
            if (hipError_t e = hipEventSynchronize(ring.moved[slot]); e != hipSuccess) return t.fail(e);
            memcpy(to + c * kRingChunk, ring.slot[slot], size_of(c));
            t.host_done[slot].store(c + 1, std::memory_order_release);
        }
    };
    if (chunks == 1) {
        drive();
        empty(0, 1);
        return hipError_t(t.error.load());
    }
    return run_transfer(t, chunks, empty, drive);
}

}  // namespace itak
