"""csrc/ring_cut.h on the CPU: the chunks of a transfer through the pinned ring."""
import os
import subprocess

import pytest

from helpers import ROOT

PROGRAM = r"""
#include "ring_cut.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
using namespace itak;
int main(int argc, char **argv) {
    const RampAt at = !strcmp(argv[1], "first") ? RampAt::First : !strcmp(argv[1], "many") ? RampAt::FirstOfMany : RampAt::Last;
    for (int i = 2; i < argc; ++i) {
        ring_cut(strtoull(argv[i], nullptr, 0), at, [](uint64_t from, uint64_t n) { printf("%llu,%llu ", (unsigned long long)from, (unsigned long long)n); });
        printf("\n");
    }
}
"""
MB = 1 << 20


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    folder = tmp_path_factory.mktemp("cut")
    src, exe = folder / "cut.cpp", folder / "cut"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "itak-torch-rebuild_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    return lambda ramp, size: [tuple(map(int, x.split(",")))
                               for x in subprocess.run([str(exe), ramp, str(size)], capture_output=True, text=True).stdout.split()]


# Whole chunks up to which a transfer is not cut finer: four, eight for uploads of bytes as they lie.
@pytest.mark.parametrize("ramp,plain", [("first", 4), ("last", 4), ("many", 8)])
@pytest.mark.parametrize("size", [4, 4 * MB - 4, 4 * MB, 4 * MB + 4, 16 * MB, 16 * MB + 4, 17 * MB, 32 * MB, 32 * MB + 4, 33 * MB,
                                  100 * MB + 12])
def test_chunks_cover_a_transfer_in_order(cut, ramp, plain, size):
    chunks = cut(ramp, size)
    at = 0
    for start, n in chunks:
        assert start == at and 0 < n <= 4 * MB and start // (4 * MB) == (start + n - 1) // (4 * MB)
        at += n
    assert at == size
    whole = -(-size // (4 * MB))
    if whole <= plain:
        assert len(chunks) == whole
    else:
        for start, n in chunks:  # units of 4 MB from the end that is cut
            unit = start // (4 * MB) if ramp != "last" else whole - 1 - start // (4 * MB)
            part = {0: MB, 1: 2 * MB}.get(unit, 4 * MB)
            assert n == min(part, size - start)
