"""Chunks of a prompt around the lines of their two planners: the chunk append (runs from 64 rows on,
any first row, rings that wrap inside the run) against the row kernel, raw plane for raw plane, and the
block kernel's choice of tiles and splits (behind its own append up to 64 rows, one tile or two beyond)
against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("window", [None, 96])
@pytest.mark.parametrize("d", [128, 80])
@pytest.mark.parametrize("first", [0, 1, 31, 32, 77])
@pytest.mark.parametrize("rows", [64, 65, 96, 127, 200])
def test_chunk_append_writes_what_the_row_kernel_writes(rows, first, d, window):
    P = pkg()
    kv_heads = 3
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    rng = np.random.default_rng(rows * 100 + first)
    k, v = normal(rng, first + rows, kv_heads * d), normal(rng, first + rows, kv_heads * d)
    k[first + 2, 3], v[first + 3, 5] = np.nan, np.inf
    kd, vd = dev(k), dev(v)
    planes = []
    for piece in (rows, 50):
        pool = P.KvPool([kind], kv_heads, d, elem="f16", max_slots=2, capacity_rows=320, ring_headroom=200)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        pool.acquire()
        cache = pool.acquire()
        at = 0
        while at < first + rows:
            n = min(50, first - at) if at < first else min(piece, first + rows - at)
            pool.append_device(0, [(cache, n)], kd[at:].data_ptr(), vd[at:].data_ptr())
            at += n
        torch.cuda.synchronize()
        planes.append(cache.read_raw(0))
        pool.close()
    for got, want in zip(*planes):
        assert np.array_equal(np.asarray(got).view(np.uint8), np.asarray(want).view(np.uint8))


@pytest.mark.parametrize("window", [None, 300])
@pytest.mark.parametrize("q_heads,kv_heads", [(32, 4), (8, 1), (10, 2)])
@pytest.mark.parametrize("rows,ctx", [(63, 700), (65, 0), (65, 1300), (129, 70), (257, 1300), (520, 400), (700, 33)])
def test_chunks_against_the_oracle(rows, ctx, q_heads, kv_heads, window):
    P = pkg()
    d = 128
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    rng = np.random.default_rng(rows + ctx)
    pool = P.KvPool([kind], kv_heads, d, elem="f16", capacity_rows=ctx + rows, ring_headroom=max(64, rows))
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    cache = pool.acquire()
    ref = oracle.KvCache.new([okind], kv_heads, d, store_f16=True)
    k, v = normal(rng, ctx + rows, kv_heads * d), normal(rng, ctx + rows, kv_heads * d)
    kd, vd = dev(k), dev(v)
    for at in range(0, ctx, 50):
        pool.append_device(0, [(cache, min(50, ctx - at))], kd[at:].data_ptr(), vd[at:].data_ptr())
    for i in range(ctx):
        ref.append(0, k[i], v[i], i)
    q = normal(rng, rows, q_heads * d)
    qd = dev(q)
    out = torch.empty_like(qd)
    pool.attention_step_device(0, [(cache, rows)], qd.data_ptr(), kd[ctx:].data_ptr(), vd[ctx:].data_ptr(),
                               out.data_ptr(), q_heads)
    torch.cuda.synchronize()
    want = oracle.attention_step(ref, 0, q, k[ctx:], v[ctx:], q_heads, ctx, threads=8)
    assert max_abs(out.cpu().numpy().reshape(-1), want) <= 2e-3
    pool.close()


# The block kernel at its other head dims, whose plans are priced by figures of their own: few and many rows,
# short runs and long ones, one and several items. The allocation-free call takes the best plan its workspace
# holds.
@pytest.mark.parametrize("window", [None, 200])
@pytest.mark.parametrize("q_heads,kv_heads", [(32, 4), (8, 1), (6, 3)])
@pytest.mark.parametrize("rows,ctx", [(9, 40), (7, 420), (17, 600), (40, 1500), (130, 300), (60, 3900)])
@pytest.mark.parametrize("d", [64, 96, 256])
def test_blocks_at_the_other_head_dims(d, rows, ctx, q_heads, kv_heads, window):
    P = pkg()
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    rng = np.random.default_rng(rows + ctx + d)
    contexts, width = (ctx, ctx // 5), kv_heads * d
    refs = [oracle.KvCache.new([okind], kv_heads, d, store_f16=True) for _ in contexts]
    pools = [P.KvPool([kind], kv_heads, d, elem="f16", max_slots=2, capacity_rows=ctx + rows, ring_headroom=max(64, rows))
             for _ in range(2)]
    caches = [[pool.acquire() for _ in contexts] for pool in pools]
    for s, n in enumerate(contexts):
        first = 0 if window is None else max(0, n - window)
        k, v = normal(rng, n - first, width), normal(rng, n - first, width)
        for cache in (caches[0][s], caches[1][s], refs[s]):
            cache.restore_bulk(0, first, k, v)
    q, k, v = (normal(rng, 2 * rows, w) for w in (q_heads * d, width, width))
    qd, kd, vd = dev(q), dev(k), dev(v)
    want = np.concatenate([np.asarray(oracle.attention_step(refs[s], 0, q[s * rows:][:rows], k[s * rows:][:rows],
                                                            v[s * rows:][:rows], q_heads, contexts[s], threads=8)).reshape(-1)
                           for s in range(2)])
    for pool, held, step in zip(pools, caches, ("attention_step_device", "attention_step_device_noalloc")):
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        out = torch.full_like(qd, float("nan"))
        getattr(pool, step)(0, [(c, rows) for c in held], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
        torch.cuda.synchronize()
        assert max_abs(out.cpu().numpy().reshape(-1), want) <= 2e-3, step
        pool.close()
