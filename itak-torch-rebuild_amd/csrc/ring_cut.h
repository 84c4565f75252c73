// How a transfer through the pinned ring (host_ring.h) is cut into chunks. Plain C++, without the runtime.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace itak {

constexpr uint64_t kRingChunk = 4ull << 20;
constexpr uint32_t kRingSlots = 8;

// `bytes` bytes cut into chunks of kRingChunk, one at the end that the link waits for in four and its neighbour in two:
// the first of an upload, the last of a download. fn(at, n) for each in order. Runs of few chunks stay as they are: every
// chunk more is a helper more to start, and a single chunk is moved by the calling thread (1.9 MB loaded 231 us in one,
// 264 in two). Uploads of bytes as they lie only from nine chunks on: up to eight are a thread each, and version 2
// loads took 4 % longer with theirs cut (16 layers of 520 / 700 rows, least of 50, 0.87 / 1.00 -> 0.83 / 0.96 ms); halves, which are narrowed on the way, from five.
enum class RampAt { First, FirstOfMany, Last };
template <class F>
void ring_cut(uint64_t bytes, RampAt ramp_at, F fn) {
    const uint64_t unit = kRingChunk, whole = (bytes + unit - 1) / unit;
    const bool ramp = whole > (ramp_at == RampAt::FirstOfMany ? kRingSlots : kRingSlots / 2);
    for (uint64_t c = 0; c < whole; ++c) {
        const uint64_t from_end = ramp_at != RampAt::Last ? c : whole - 1 - c;
        const uint64_t part = unit / (!ramp ? 1 : from_end == 0 ? 4 : from_end == 1 ? 2 : 1);
        const uint64_t end = std::min(bytes, (c + 1) * unit);
        for (uint64_t at = c * unit; at < end; at += part) fn(at, std::min(part, end - at));
    }
}

}  // namespace itak
