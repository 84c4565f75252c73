// Host code: see host_ring.h.
#include "host_ring.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <thread>

#include "host_halves.h"
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

// Part of a transfer that goes through one slot: bytes [at, at + bytes) of it.
struct Chunk {
    const unsigned char *src;
    unsigned char *dst;
    uint64_t bytes;
    uint64_t at;
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

// The upload of `chunks`: fill_slot(c, slot memory) on the helpers, send(c, slot memory) on this thread, in order.
template <class Fill, class Send>
hipError_t run_upload(HostRing &ring, uint64_t chunks, hipStream_t stream, Fill fill_slot, Send send) {
    if (chunks == 0) return hipSuccess;
    if (hipError_t e = ring.open(chunks); e != hipSuccess) return e;
    Transfer t;
    auto fill = [&](uint64_t first, uint64_t step) {
        for (uint64_t c = first; c < chunks; c += step) {
            const uint32_t slot = c % kRingSlots;
            if (c >= kRingSlots) {
                if (!t.wait([&] { return t.enqueued.load(std::memory_order_acquire) > c - kRingSlots; })) return;
                if (hipError_t e = hipEventSynchronize(ring.moved[slot]); e != hipSuccess) return t.fail(e);
            }
            fill_slot(c, ring.slot[slot]);
            t.host_done[slot].store(c + 1, std::memory_order_release);
        }
    };
    auto drive = [&] {
        for (uint64_t c = 0; c < chunks; ++c) {
            const uint32_t slot = c % kRingSlots;
            if (!t.wait([&] { return t.host_done[slot].load(std::memory_order_acquire) == c + 1; })) return;
            hipError_t e = send(c, ring.slot[slot], ring.moved[slot], t.enqueued);
            if (e != hipSuccess) return t.fail(e);
        }
    };
    if (chunks == 1) {  // nothing to overlap
        fill(0, 1);
        drive();
        return hipError_t(t.error.load());
    }
    return run_transfer(t, chunks, fill, drive);
}

}  // namespace

bool host_has_f16() {
    static const bool has = has_f16c();
    return has;
}

hipError_t ring_upload(HostRing &ring, const std::vector<RingSpan> &spans, hipStream_t stream,
                       const std::function<hipError_t(uint64_t)> &after) {
    std::vector<Chunk> chunks;
    for (size_t i = 0; i < spans.size(); ++i) {
        const RingSpan &s = spans[i];
        const auto add = [&](uint64_t at, uint64_t n) {
            chunks.push_back(Chunk{static_cast<const unsigned char *>(s.src) + at, static_cast<unsigned char *>(s.dst) + at, n, at});
        };
        if (i == 0)
            ring_cut(s.bytes, RampAt::FirstOfMany, add);
        else
            for (uint64_t at = 0; at < s.bytes; at += kRingChunk) add(at, std::min(kRingChunk, s.bytes - at));
    }
    uint64_t sent = 0;
    return run_upload(
        ring, chunks.size(), stream, [&](uint64_t c, unsigned char *slot) { memcpy(slot, chunks[c].src, chunks[c].bytes); },
        [&](uint64_t c, unsigned char *slot, hipEvent_t moved, std::atomic<uint64_t> &enqueued) {
            hipError_t e = hipMemcpyAsync(chunks[c].dst, slot, chunks[c].bytes, hipMemcpyHostToDevice, stream);
            if (e == hipSuccess) e = hipEventRecord(moved, stream);
            sent += chunks[c].bytes;
            if (e == hipSuccess) enqueued.store(c + 1, std::memory_order_release);
            return e == hipSuccess && after ? after(sent) : e;
        });
}

hipError_t ring_upload_narrow(HostRing &ring, const void *src, uint64_t bytes, void *floats, void *halves, hipStream_t stream,
                              const std::function<hipError_t(uint64_t, uint64_t, uint64_t)> &after) {
    std::vector<Chunk> chunks;
    ring_cut(bytes, RampAt::First, [&](uint64_t at, uint64_t n) {
        chunks.push_back(Chunk{static_cast<const unsigned char *>(src) + at, static_cast<unsigned char *>(floats) + at, n, at});
    });
    // One value that is no f16's says what the rest holds: no thread tries any further.
    std::atomic<bool> worth_it{true};
    std::vector<unsigned char> narrowed(chunks.size(), 0);
    uint64_t from = 0, to = 0;  // arrived as halves and not reported
    return run_upload(
        ring, chunks.size(), stream,
        [&](uint64_t c, unsigned char *slot) {
            narrowed[c] = narrow_chunk(slot, chunks[c].src, chunks[c].bytes, worth_it);
            if (!narrowed[c]) memcpy(slot, chunks[c].src, chunks[c].bytes);
        },
        [&](uint64_t c, unsigned char *slot, hipEvent_t moved, std::atomic<uint64_t> &enqueued) {
            const Chunk &k = chunks[c];
            void *dst = narrowed[c] ? static_cast<unsigned char *>(halves) + k.at % (kRingChunk * kRingSlots) / 2 : k.dst;
            hipError_t e = hipMemcpyAsync(dst, slot, narrowed[c] ? k.bytes / 2 : k.bytes, hipMemcpyHostToDevice, stream);
            if (e == hipSuccess) e = hipEventRecord(moved, stream);
            if (e != hipSuccess) return e;
            enqueued.store(c + 1, std::memory_order_release);
            if (narrowed[c] && to == k.at) {
                to = k.at + k.bytes;
            } else if (narrowed[c]) {  // behind a chunk that came as floats: what lay before it goes first
                if (to > from) e = after(k.at, from, to);
                from = k.at, to = k.at + k.bytes;
            }
            if (e != hipSuccess) return e;
            const uint64_t end = k.at + k.bytes;
            if (end < bytes && end % (kRingChunk * kRingSlots) != 0) return hipSuccess;
            e = after(end, from, to);
            from = to = end;
            return e;
        });
}

hipError_t ring_download(HostRing &ring, void *out, uint64_t bytes, hipStream_t stream, bool widen,
                         const std::function<hipError_t(uint64_t, uint64_t, const void **)> &source) {
    if (bytes == 0) return hipSuccess;
    std::vector<Chunk> list;
    ring_cut(bytes, RampAt::Last, [&](uint64_t at, uint64_t n) {
        list.push_back(Chunk{nullptr, static_cast<unsigned char *>(out) + at, n, at});
    });
    const uint64_t chunks = list.size();
    if (hipError_t e = ring.open(chunks); e != hipSuccess) return e;
    Transfer t;
    auto drive = [&] {
        for (uint64_t c = 0; c < chunks; ++c) {
            const uint32_t slot = c % kRingSlots;
            if (c >= kRingSlots &&
                !t.wait([&] { return t.host_done[slot].load(std::memory_order_acquire) == c - kRingSlots + 1; }))
                return;
            const void *from = nullptr;
            hipError_t e = source(list[c].at, list[c].bytes, &from);
            if (e == hipSuccess)
                e = hipMemcpyAsync(ring.slot[slot], from, widen ? list[c].bytes / 2 : list[c].bytes, hipMemcpyDeviceToHost, stream);
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
            if (widen)
                widen_halves(list[c].dst, ring.slot[slot], list[c].bytes);
            else
                memcpy(list[c].dst, ring.slot[slot], list[c].bytes);
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
