"""Host-pointer attention calls return when the last word of their output has arrived, which the launch
that made it may outlast; csrc/host_turns.h decides which half of the pinned staging the next call packs
into and when launches must have ended first.

On the CPU: the class itself under random calls, failures and changes of stream, against a device that
keeps every launch running for as long as it may. On the GPU: calls whose stored rows are fetched behind
the output, back to back, and a change of stream right after a call; rows bit for bit. And caches with
a pool of their own, in turn and from several threads, which leave their staging to each other."""
import os
import subprocess
import threading

import numpy as np
import pytest

import oracle
from helpers import ROOT, normal, pkg, rel_err

PROGRAM = r"""
#include "host_turns.h"
#include <cstdio>
#include <cstdlib>
using itak::HostTurns;
// A call's launches read its half until they have ended: at the latest when the next call on the same
// stream is seen, or when its stream is waited for.
struct Reader { bool live; int stream; } reader[2];
static char streams[3];
int main(int argc, char **argv) {
    unsigned x = unsigned(atoi(argv[1]));
    auto random = [&](unsigned n) { x = x * 1664525u + 1013904223u; return (x >> 16) % n; };
    for (int round = 0; round < 2000; ++round) {
        HostTurns turns;
        reader[0] = reader[1] = Reader{false, 0};
        int stream = 0;
        auto wait = [&](int s) { for (Reader &r : reader) if (r.stream == s) r.live = false; };
        for (int step = 0; step < 60; ++step) {
            const unsigned what = random(8);
            if (what == 0) {  // another stream; the pool waits unless one of the two is captured
                const int next = int(random(3));
                if (next != stream && turns.running() && random(2)) {
                    wait(int(static_cast<const char *>(turns.stream()) - streams));
                    turns.drained();
                }
                stream = next;
                continue;
            }
            if (turns.must_drain(streams + stream)) {
                wait(int(static_cast<const char *>(turns.stream()) - streams));
                turns.drained();
            }
            const unsigned half = turns.begin(streams + stream);
            if (half > 1) return 2;
            if (reader[half].live) { printf("round %d step %d: half %u is still read\n", round, step, half); return 1; }
            for (Reader &r : reader) if (r.live && r.stream != stream) { printf("a reader on another stream\n"); return 1; }
            if (what == 1) { if (random(2)) reader[half] = Reader{true, stream}; continue; }  // fails before or after a launch
            reader[half] = Reader{true, stream};
            // Output seen: what ran on the stream before this call's launches has ended.
            reader[half ^ 1].live = false;
            if (what == 2) { wait(stream); turns.drained(); } else turns.seen();
        }
    }
    return 0;
}
"""


def test_no_half_is_packed_while_a_launch_may_read_it(tmp_path):
    src, exe = tmp_path / "turns.cpp", tmp_path / "turns"
    src.write_text(PROGRAM)
    include = os.path.join(ROOT, "itak-torch-rebuild_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", include, str(src), "-o", str(exe)], check=True)
    for seed in range(8):
        done = subprocess.run([str(exe), str(seed)], capture_output=True, text=True)
        assert done.returncode == 0, (seed, done.stdout)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [17, 20, 25])  # on eight wavefronts, of which four write no output at head_dim 64
def test_rows_fetched_behind_the_output_are_the_calls_own(rows):
    import torch

    P = pkg()
    rng = np.random.default_rng(rows)
    q_heads, kv_heads, d, ctx, calls = 8, 1, 64, 100, 24
    pool = P.KvPool(1, kv_heads, d, elem="f32", max_slots=1, capacity_rows=ctx + calls * rows)
    streams = [torch.cuda.Stream() for _ in range(2)]
    pool.set_stream(streams[0].cuda_stream)
    compute, position = P.HipCompute(elem="f32", pool=pool), P.PositionCache()
    cfg = P.GlimmerConfig(layers=[P.LayerKind.Global], q_heads=q_heads, kv_heads=kv_heads, key_length=d,
                          value_length=d, sliding_window=0)
    ref = oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d)
    blocks = [ctx] + [rows] * calls
    data = [tuple(normal(rng, n, w) for w in (q_heads * d, kv_heads * d, kv_heads * d)) for n in blocks]
    outs = []
    for i, (n, (q, k, v)) in enumerate(zip(blocks, data)):
        outs.append(compute.attention(P.AttentionRequest(q, k, v, 0, P.LayerKind.Global, cfg), position))
        position.advance(n)
        if i % 5 == 4:
            pool.set_stream(streams[i // 5 % 2].cuda_stream)
    for n, (q, k, v), out in zip(blocks, data, outs):
        want = oracle.attention_step(ref, 0, q, k, v, q_heads, ref.next_position(0), oracle.AttentionParams(), threads=8)
        assert rel_err(np.asarray(out).reshape(-1), want) <= 1e-5
    total = ctx + calls * rows
    _, keys, values = compute.kv_cache().read_rows(0, 0, total)
    for side, got in ((1, keys), (2, values)):
        want = np.concatenate([x[side] for x in data])
        assert np.asarray(got).tobytes() == want.tobytes()
    pool.synchronize()
    pool.close()


@pytest.mark.gpu
def test_caches_of_their_own_in_turn_and_from_threads():
    P = pkg()
    q_heads, kv_heads, d = 8, 2, 64
    failed = []

    def sequences(seed, count):
        try:
            rng = np.random.default_rng(seed)
            for i in range(count):
                n, nq = int(rng.integers(20, 200)), int(rng.integers(1, 400 if i == 2 else 12))  # (one staging outgrows the rest)
                nq = min(nq, n)
                k, v, q = (normal(rng, n, kv_heads * d), normal(rng, n, kv_heads * d), normal(rng, nq, q_heads * d))
                cache = P.KvCache.new([P.LayerKind.Global], kv_heads, d, elem="f32", capacity_rows=256)
                ref = oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d)
                cache.restore_bulk(0, 0, k, v)
                ref.restore_bulk(0, 0, k, v)
                at = list(range(n - nq, n))
                for _ in range(2):
                    got = P.gqa_attention(q, nq, q_heads, at, cache.view(0), P.AttentionParams())
                    want = oracle.gqa_attention(q, nq, q_heads, at, ref.view(0), oracle.AttentionParams())
                    assert rel_err(np.asarray(got).reshape(-1), np.asarray(want).reshape(-1)) <= 1e-5, (seed, i)
                cache.pool.close()
        except BaseException as e:  # noqa: B036 - reported by the main thread
            failed.append((seed, repr(e)))

    sequences(0, 6)
    threads = [threading.Thread(target=sequences, args=(seed, 8)) for seed in range(1, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
