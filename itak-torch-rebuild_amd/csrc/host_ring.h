// Moving bytes between ordinary host memory and the device through a ring of pinned slots.
//
// The runtime's own copy from or to pageable memory is one thread's memcpy in front of the link
// (8 to 10 GB/s on this host, less where the destination's pages are touched for the first time),
// and the link carries 55 GB/s. Here up to eight host threads fill or empty the slots while the
// copy engine works on others, in the order of the stream. 4 MiB a slot: a copy command costs
// microseconds and 4 MiB take 75 on the link; eight slots keep eight threads busy.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <vector>

namespace itak {

constexpr uint64_t kRingChunk = 4ull << 20;
constexpr uint32_t kRingSlots = 8;

struct HostRing {
    unsigned char *slot[kRingSlots] = {};  // pinned, kRingChunk bytes each
    hipEvent_t moved[kRingSlots] = {};     // behind the last copy from or to the slot
    hipError_t open(uint64_t slots);       // makes the first `slots` slots usable; keeps what it has
    void close();
};

struct RingSpan {
    const void *src;
    void *dst;
    uint64_t bytes;
};

// Host spans to device spans, enqueued on `stream` in order; `after(n)`, when given, is called on
// the calling thread whenever the copies of the first n bytes (of all spans together) have been
// enqueued. Returns with copies in flight: the slots are free again once the stream has passed.
hipError_t ring_upload(HostRing &ring, const std::vector<RingSpan> &spans, hipStream_t stream,
                       const std::function<hipError_t(uint64_t)> &after = nullptr);

// `bytes` bytes to host memory at `out`, chunk by chunk: `source(at, n, &p)` enqueues whatever
// makes bytes [at, at + n) on the stream and says where they lie in device memory; `at` goes up in
// steps of kRingChunk. Returns when the bytes are in place.
hipError_t ring_download(HostRing &ring, void *out, uint64_t bytes, hipStream_t stream,
                         const std::function<hipError_t(uint64_t, uint64_t, const void **)> &source);

}  // namespace itak
