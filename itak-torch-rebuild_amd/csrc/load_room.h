// What loading a snapshot holds in device memory beside the pool. Plain C++, without the runtime.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace itak {

// One allocation: the payload's n bytes, the checksum's state, the sum's scratch, and, where f32 rows cross the link
// as halves, a place for one piece's halves, which the stream reads before the next piece's come.
struct LoadRoom {
    uint64_t state_at = 0, scratch_at = 0, halves_at = 0, halves_bytes = 0, bytes = 0;
};
inline LoadRoom load_room(uint64_t n, uint64_t piece, uint64_t sum_scratch, bool halves) {
    const auto up = [](uint64_t x) { return (x + 255) / 256 * 256; };
    LoadRoom r;
    r.state_at = up(n);
    r.scratch_at = r.state_at + 256;
    r.halves_at = r.scratch_at + up(sum_scratch);
    r.halves_bytes = halves ? up(std::min(n, piece)) / 2 : 0;
    r.bytes = r.halves_at + r.halves_bytes;
    return r;
}
// The room that `make(bytes)` grants: with a place for halves when `halves` asks for one, without when that is too much.
template <class Make>
bool take_load_room(uint64_t n, uint64_t piece, uint64_t sum_scratch, bool halves, Make make, LoadRoom &out) {
    out = load_room(n, piece, sum_scratch, halves);
    if (make(out.bytes)) return true;
    if (!halves) return false;
    out = load_room(n, piece, sum_scratch, false);
    return make(out.bytes);
}

}  // namespace itak
