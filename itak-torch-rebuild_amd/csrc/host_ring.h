// Moving bytes between ordinary host memory and the device through a ring of pinned slots.
//
// The runtime's own copy from or to pageable memory is one thread's memcpy in front of the link
// (8 to 10 GB/s on this host, less where the destination's pages are touched for the first time),
// and the link carries 55 GB/s. Here up to eight host threads fill or empty the slots while the
// copy engine works on others, in the order of the stream. 4 MiB a slot: a copy command costs
// ten microseconds and 4 MiB take 75 on the link; eight slots keep eight threads busy. A thread takes a few
// hundred microseconds over 4 MiB, though, so an upload begins and a download ends with smaller chunks.
//
// Rows that are f32 outside and f16 values inside cross the link as halves: the host threads widen them
// as they empty a slot (f16 to f32 is exact), or narrow them as they fill one where every value of the chunk
// is an f16's, and the device narrows or widens on its side. The link then carries half the bytes, and
// what the threads read and write is a quarter less.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <vector>

#include "ring_cut.h"

namespace itak {

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

// f32 values at `src` to device memory, as halves (16-byte aligned) while every value is an f16's, else as they are at
// floats + at. The halves of each kRingChunk * kRingSlots bytes of values take the place of the last ones', at halves +
// at % (kRingChunk * kRingSlots) / 2: `after(n, from, to)` is called like ring_upload's and at the end of each such
// piece, with the bytes [from, to) (of the f32 values) that have arrived as halves since the last call, all others among
// them as floats, and what it enqueues reads them before the next ones come.
hipError_t ring_upload_narrow(HostRing &ring, const void *src, uint64_t bytes, void *floats, void *halves, hipStream_t stream,
                              const std::function<hipError_t(uint64_t, uint64_t, uint64_t)> &after);
// Whether this host converts halves in its vector units (both calls that do need it).
bool host_has_f16();

// `bytes` bytes to host memory at `out`, chunk by chunk: `source(at, n, &p)` enqueues whatever
// makes bytes [at, at + n) on the stream and says where they lie in device memory; `at` goes up in
// steps of at most kRingChunk, and no step crosses a multiple of it. `widen`: the device holds halves, and f32
// values are wanted (`at`, `n` and `bytes` count those). Returns when the bytes are in place.
hipError_t ring_download(HostRing &ring, void *out, uint64_t bytes, hipStream_t stream, bool widen,
                         const std::function<hipError_t(uint64_t, uint64_t, const void **)> &source);

}  // namespace itak
