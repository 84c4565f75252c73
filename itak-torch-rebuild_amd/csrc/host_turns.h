// Which half of the pinned staging a host-pointer attention call packs its inputs into, and when
// launches must have ended before it may. Plain C++, without the runtime.
//
// Such a call may return when the last word of its output has arrived, and its last launch is then
// still allowed to read the inputs (a workgroup that copies new rows to the planes behind its output) and
// to store rows. So the next call packs into the other half, and by the time a half's turn comes again the
// call in between has been seen: its output was made by a launch behind, on the same stream, the one that
// read this half. Where that does not hold (the calls ran on different streams, or one failed before its
// output was seen) the caller waits for the launches first.
#pragma once

#include <cstdint>

namespace itak {

class HostTurns {
  public:
    // Whether launches of earlier calls must have ended before a call on `stream` packs its inputs.
    bool must_drain(const void *stream) const { return open_ || (running_ && stream_ != stream); }
    // Whether launches of earlier calls may still be running, and the stream they are on.
    bool running() const { return running_; }
    const void *stream() const { return stream_; }
    // A call begins on `stream`: the half it packs into.
    uint32_t begin(const void *stream) {
        open_ = running_ = true;
        stream_ = stream;
        return half_ ^= 1u;
    }
    // Its output arrived, made by its last launch.
    void seen() { open_ = false; }
    // Everything launched so far has ended.
    void drained() { open_ = running_ = false; }

  private:
    uint32_t half_ = 1;
    bool open_ = false;     // a call began and its output has not been seen
    bool running_ = false;
    const void *stream_ = nullptr;
};

}  // namespace itak
