"""csrc/host_halves.h, which the rows of version 1 snapshots pass on their way over the host link, on the CPU: halves and
f32 values there and back, and where narrowing gives up."""
import os
import subprocess

import numpy as np
import pytest

from helpers import ROOT

PROGRAM = r"""
#include "host_halves.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace itak;
// argv: number of values, index of a value that is no half (-1: none), its bits, whether another thread has met one.
int main(int argc, char **argv) {
    if (!has_f16c()) return 77;
    const long count = atol(argv[1]), bad = atol(argv[2]);
    std::vector<uint16_t> halves(count + 1), back(count + 1, 0xeeee);
    std::vector<float> floats(count + 1);
    for (long i = 0; i < count; ++i) halves[i] = uint16_t((i * 7919u) % 0x7c00u | (i & 1 ? 0x8000u : 0u));  // (no infinity, no NaN)
    auto bytes = [](void *p) { return static_cast<unsigned char *>(p); };
    widen_halves(bytes(floats.data()), bytes(halves.data()), count * 4);
    for (long i = 0; i < count; ++i) {  // against the value itself
        const uint16_t h = halves[i];
        const int e = h >> 10 & 31, m = h & 1023;
        double want = e ? (1024 + m) * 1.0 : m * 1.0;
        for (int x = e ? e : 1; x < 25; ++x) want *= 0.5;
        for (int x = 25; x < e; ++x) want *= 2.0;
        if (double(floats[i]) != (h & 0x8000 ? -want : want)) { printf("value %ld\n", i); return 1; }
    }
    if (bad >= 0) {
        const uint32_t bits = uint32_t(strtoul(argv[3], nullptr, 0));
        memcpy(&floats[bad], &bits, 4);
    }
    std::atomic<bool> worth_it{atol(argv[4]) == 0};
    const bool all = narrow_chunk(bytes(back.data()), bytes(floats.data()), count * 4, worth_it);
    long touched = count;
    while (touched && back[touched - 1] == 0xeeee) --touched;
    if (back[count] != 0xeeee) { printf("beyond the end\n"); return 1; }
    if (all && memcmp(back.data(), halves.data(), count * 2)) { printf("halves differ\n"); return 1; }
    printf("%d %d %ld\n", int(all), int(worth_it.load()), touched);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    folder = tmp_path_factory.mktemp("halves")
    src, exe = folder / "halves.cpp", folder / "halves"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "itak-torch-rebuild_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)

    def run(*args):
        done = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True)
        if done.returncode == 77:
            pytest.skip("this CPU has no F16C")
        assert done.returncode == 0, (args, done.stdout)
        return tuple(map(int, done.stdout.split()))
    return run


@pytest.mark.parametrize("count", [1, 7, 8, 9, 4095, 4096, 4097, 8191, 1 << 20])
def test_halves_there_and_back(program, count):
    assert program(count, -1, 0, 0) == (1, 1, count)


# The first value between two halves, beyond the largest, a NaN, a subnormal f32; the narrowing stops within 32 KB of it.
@pytest.mark.parametrize("bits", [0x3f800001, 0x477ff000, 0x7fc00000, 0x7f800001, 0x80000123])
@pytest.mark.parametrize("count,bad", [(1, 0), (9, 8), (4096, 4095), (5000, 4096), (1 << 20, 0), (1 << 20, 9), (1 << 20, 600000),
                                       (1 << 20, (1 << 20) - 1)])
def test_narrowing_stops_at_a_value_that_is_no_half(program, count, bad, bits):
    whole, worth_it, touched = program(count, bad, hex(bits), 0)
    assert (whole, worth_it) == (0, 0)
    assert touched <= (bad // 8192 + 1) * 8192


def test_narrowing_stops_when_another_thread_has_met_one(program):
    assert program(1 << 20, -1, 0, 1) == (0, 0, 0)


def test_values_between_halves_are_what_numpy_says_they_are():
    for bits in (0x3f800001, 0x477ff000, 0x80000123):
        x = np.array([bits], dtype=np.uint32).view(np.float32)
        with np.errstate(over="ignore"):
            assert x.astype(np.float16).astype(np.float32)[0] != x[0]
