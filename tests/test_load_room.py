"""csrc/load_room.h on the CPU: what loading a snapshot allocates on the device. A place for halves is one piece's, and a
device that cannot give it still gives what a load without halves takes."""
import os
import subprocess

from helpers import ROOT

PROGRAM = r"""
#include "load_room.h"
#include <cstdio>
#include <vector>
using namespace itak;
#define CHECK(x) if (!(x)) { printf("%s, n %llu\n", #x, (unsigned long long)n); return 1; }
int main() {
    const uint64_t piece = 32ull << 20, scratch = 70000;
    for (uint64_t n : {131072ull, 131076ull, 3145728ull, 33554428ull, 33554432ull, 33554436ull, 67108868ull, 5000000004ull}) {
        const LoadRoom plain = load_room(n, piece, scratch, false), both = load_room(n, piece, scratch, true);
        // The parts lie apart, in order, 256-byte aligned, and hold what goes there.
        for (const LoadRoom &r : {plain, both}) {
            CHECK(r.state_at >= n && r.scratch_at >= r.state_at + 8 && r.halves_at >= r.scratch_at + scratch);
            CHECK(r.state_at % 256 == 0 && r.scratch_at % 256 == 0 && r.halves_at % 256 == 0);
            CHECK(r.bytes == r.halves_at + r.halves_bytes);
        }
        CHECK(plain.halves_bytes == 0 && both.halves_bytes >= (n < piece ? n : piece) / 2);
        CHECK(both.bytes <= plain.bytes + piece / 2);
        // A device with `free` bytes left: the larger room, the plain one, none.
        for (uint64_t free : {both.bytes, both.bytes - 1, plain.bytes, plain.bytes - 1}) {
            std::vector<uint64_t> asked;
            const auto make = [&](uint64_t want) { asked.push_back(want); return want <= free; };
            LoadRoom got;
            const bool ok = take_load_room(n, piece, scratch, true, make, got);
            CHECK(ok == (free >= plain.bytes));
            if (ok) CHECK(asked.back() == got.bytes && got.bytes <= free && (got.halves_bytes != 0) == (free >= both.bytes));
            asked.clear();
            CHECK(take_load_room(n, piece, scratch, false, make, got) == (free >= plain.bytes));
            CHECK(asked.size() == 1 && got.halves_bytes == 0);
        }
    }
    return 0;
}
"""


def test_a_load_holds_its_payload_and_one_piece_of_halves(tmp_path):
    src, exe = tmp_path / "room.cpp", tmp_path / "room"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "itak-torch-rebuild_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
