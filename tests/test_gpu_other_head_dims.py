"""Head dims and groups that only the f32-arithmetic matrix kernel takes: both plane layouts of f16
pools and the rows of f32 pools, at the edges of its padded head dims, with groups above 16, on
global and windowed layers; decode rows and short blocks that it appends itself, longer ones behind
the append launch. f32 arithmetic over the stored rows on f16 pools too, so both are held to 1e-5 of
the oracle's largest output, and what it stores is compared bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import normal, pkg, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [
    # blocked f16 planes
    ("f16", 16, 8, 4), ("f16", 48, 6, 2), ("f16", 80, 32, 8), ("f16", 112, 5, 1), ("f16", 144, 8, 2),
    ("f16", 176, 4, 4), ("f16", 192, 12, 2), ("f16", 208, 7, 1), ("f16", 240, 8, 1),
    ("f16", 128, 66, 1), ("f16", 64, 34, 2), ("f16", 256, 17, 1), ("f16", 96, 24, 1),  # groups above 16
    # row-major f16 planes
    ("f16", 4, 4, 2), ("f16", 40, 8, 2), ("f16", 72, 9, 3), ("f16", 100, 4, 1), ("f16", 188, 8, 2), ("f16", 252, 3, 1),
    # f32 pools
    ("f32", 4, 2, 2), ("f32", 80, 32, 8), ("f32", 96, 8, 2), ("f32", 112, 20, 1), ("f32", 132, 6, 2),
    ("f32", 192, 8, 1), ("f32", 256, 16, 4),
]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("window", [None, 100])
@pytest.mark.parametrize("elem,d,q_heads,kv_heads", SHAPES)
def test_steps_against_the_oracle(elem, d, q_heads, kv_heads, window):
    P = pkg()
    rng = np.random.default_rng(d * 100 + q_heads)
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    pool = P.KvPool([kind], kv_heads, d, elem=elem, max_slots=2, capacity_rows=1100, ring_headroom=160)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in range(2)]
    refs = [oracle.KvCache.new([okind], kv_heads, d, store_f16=elem == "f16") for _ in range(2)]
    row = kv_heads * d
    kept = []
    for i, rows in enumerate(([150, 1], [1, 1], [1, 31], [2, 1], [160, 0], [1, 7], [1, 1], [130, 40], [1, 1], [0, 3], [65, 150], [1, 2])):
        softcap = 30.0 if i % 3 == 2 else 0.0
        total = sum(rows)
        q, k, v = normal(rng, total, q_heads * d), normal(rng, total, row), normal(rng, total, row)
        qd, kd, vd = dev(q), dev(k), dev(v)
        out = torch.empty_like(qd)
        pool.attention_step_device(0, [(c, r) for c, r in zip(caches, rows) if r], qd.data_ptr(), kd.data_ptr(),
                                   vd.data_ptr(), out.data_ptr(), q_heads, softcap=softcap)
        torch.cuda.synchronize()
        got, at = out.cpu().numpy(), 0
        for s, r in enumerate(rows):
            if r:
                base = refs[s].next_position(0)
                want = oracle.attention_step(refs[s], 0, q[at:at + r], k[at:at + r], v[at:at + r], q_heads, base,
                                             oracle.AttentionParams(softcap=softcap), threads=8)
                assert rel_err(got[at:at + r].reshape(-1), want) <= 1e-5, (rows, s, base)
                kept.append((s, base, k[at:at + r], v[at:at + r]))
                at += r
    store = (lambda x: oracle.f32_to_f16_array(x)) if elem == "f16" else (lambda x: x)
    for s, base, k, v in kept:
        oldest = caches[s].next_position(0) - caches[s].stored_len(0)
        for r in range(len(k)):
            if base + r >= oldest and (r < 3 or r > len(k) - 3):
                _, gk, gv = caches[s].read_rows(0, base + r - oldest, 1)
                assert np.array_equal(gk.reshape(-1), store(k[r]).reshape(-1)), (s, base, r)
                assert np.array_equal(gv.reshape(-1), store(v[r]).reshape(-1)), (s, base, r)
    pool.close()


@pytest.mark.parametrize("elem,d", [("f16", 80), ("f16", 40), ("f32", 96), ("f32", 192)])
@pytest.mark.parametrize("rows", [1, 4, 23])
def test_values_that_are_not_finite_reach_the_rows_that_see_them(elem, d, rows):
    P = pkg()
    q_heads, kv_heads, ctx, window = 8, 2, 70, 50
    rng = np.random.default_rng(d + rows)
    for kind, okind in ((P.LayerKind.Global, oracle.LayerKind.Global),
                        (P.LayerKind.windowed(window), oracle.LayerKind.windowed(window))):
        k, v = normal(rng, ctx + rows, kv_heads * d), normal(rng, ctx + rows, kv_heads * d)
        v[ctx + rows - 1, 3] = np.inf          # seen by the last row alone
        v[ctx - window + 1, 5] = np.nan        # on the ring: by the first rows alone
        v[ctx - window - 2, 7] = -np.inf       # on the ring: by none
        q = normal(rng, rows, q_heads * d)
        pool = P.KvPool([kind], kv_heads, d, elem=elem, capacity_rows=ctx + rows + 8)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        cache = pool.acquire()
        ref = oracle.KvCache.new([okind], kv_heads, d, store_f16=elem == "f16")
        qd, kd, vd = dev(q), dev(k), dev(v)
        for at in range(0, ctx, 35):
            pool.append_device(0, [(cache, 35)], kd[at:].data_ptr(), vd[at:].data_ptr())
        for i in range(ctx):
            ref.append(0, k[i], v[i], i)
        out = torch.empty_like(qd)
        pool.attention_step_device(0, [(cache, rows)], qd.data_ptr(), kd[ctx:].data_ptr(), vd[ctx:].data_ptr(),
                                   out.data_ptr(), q_heads)
        torch.cuda.synchronize()
        got = out.cpu().numpy().reshape(-1)
        want = np.asarray(oracle.attention_step(ref, 0, q, k[ctx:], v[ctx:], q_heads, ctx, threads=4)).reshape(-1)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isinf(got), np.isinf(want))
        fine = np.isfinite(want)
        assert (~fine).any() and rel_err(got[fine], want[fine]) <= 1e-5
        pool.close()


# Head dims of the block kernel: steps of up to 16 query vectors run here too, to f32's precision.
@pytest.mark.parametrize("window", [None, 100])
@pytest.mark.parametrize("d,q_heads,kv_heads", [(64, 32, 4), (96, 8, 8), (256, 16, 1)])
def test_short_steps_at_the_block_kernels_head_dims(d, q_heads, kv_heads, window):
    P = pkg()
    rng = np.random.default_rng(d)
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    pool = P.KvPool([kind], kv_heads, d, elem="f16", max_slots=2, capacity_rows=700)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in range(2)]
    refs = [oracle.KvCache.new([okind], kv_heads, d, store_f16=True) for _ in range(2)]
    most = 16 // (q_heads // kv_heads)
    for i, rows in enumerate(([most, 1], [1, 1], 300, [1, most], [1, 1], 300, [most, most], [1, 1])):
        if isinstance(rows, int):  # a prompt, so that contexts are split too
            k, v = normal(rng, rows, kv_heads * d), normal(rng, rows, kv_heads * d)
            kd, vd = dev(k), dev(v)
            for at in range(0, rows, 50):
                pool.append_device(0, [(caches[0], 50)], kd[at:].data_ptr(), vd[at:].data_ptr())
            for r in range(rows):
                refs[0].append(0, k[r], v[r], refs[0].next_position(0))
            continue
        softcap = 30.0 if i % 3 == 2 else 0.0
        total = sum(rows)
        q = normal(rng, total, q_heads * d)
        k, v = normal(rng, total, kv_heads * d), normal(rng, total, kv_heads * d)
        qd, kd, vd = dev(q), dev(k), dev(v)
        out = torch.empty_like(qd)
        pool.attention_step_device(0, list(zip(caches, rows)), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                   out.data_ptr(), q_heads, softcap=softcap)
        torch.cuda.synchronize()
        got, at = out.cpu().numpy(), 0
        for s, r in enumerate(rows):
            base = refs[s].next_position(0)
            want = oracle.attention_step(refs[s], 0, q[at:at + r], k[at:at + r], v[at:at + r], q_heads, base,
                                         oracle.AttentionParams(softcap=softcap), threads=8)
            assert rel_err(got[at:at + r].reshape(-1), want) <= 1e-5, (rows, s, base)
            at += r
    pool.close()


# Row-major and blocked planes on four and eight wavefronts, whole and split, rows brought along by every
# tile of a step: contexts at the ends of rounds of four, eight, sixteen and twenty-four blocks.
@pytest.mark.parametrize("elem,d,q_heads,kv_heads", [("f32", 64, 32, 4), ("f32", 128, 8, 8), ("f32", 100, 9, 3), ("f16", 80, 32, 8),
                                                     ("f16", 72, 8, 1), ("f16", 112, 40, 2)])
@pytest.mark.parametrize("ctx", [10, 60, 127, 250, 500, 760, 1500])
def test_rounds_of_wavefronts(elem, d, q_heads, kv_heads, ctx):
    P = pkg()
    rng = np.random.default_rng(d + ctx)
    pool = P.KvPool([P.LayerKind.Global], kv_heads, d, elem=elem, max_slots=2, capacity_rows=1600)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in range(2)]
    refs = [oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d, store_f16=elem == "f16") for _ in range(2)]
    for cache, ref, n in zip(caches, refs, (ctx, ctx // 3)):
        k, v = normal(rng, n, kv_heads * d), normal(rng, n, kv_heads * d)
        kd, vd = dev(k), dev(v)
        pool.append_device(0, [(cache, n)], kd.data_ptr(), vd.data_ptr())
        for i in range(n):
            ref.append(0, k[i], v[i], i)
    kept = []
    for rows in ((1, 1), (8, 3), (1, 16)):
        total = sum(rows)
        q = normal(rng, total, q_heads * d)
        k, v = normal(rng, total, kv_heads * d), normal(rng, total, kv_heads * d)
        qd, kd, vd = dev(q), dev(k), dev(v)
        out = torch.empty_like(qd)
        pool.attention_step_device(0, list(zip(caches, rows)), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
        torch.cuda.synchronize()
        got, at = out.cpu().numpy(), 0
        for s, r in enumerate(rows):
            want = oracle.attention_step(refs[s], 0, q[at:at + r], k[at:at + r], v[at:at + r], q_heads,
                                         refs[s].next_position(0), threads=8)
            assert rel_err(got[at:at + r].reshape(-1), want) <= 1e-5, (rows, s)
            kept.append((s, refs[s].next_position(0) - r, k[at:at + r], v[at:at + r]))
            at += r
    store = (lambda x: oracle.f32_to_f16_array(x)) if elem == "f16" else (lambda x: x)
    for s, base, k, v in kept:  # what the launches appended
        for r in range(len(k)):
            _, gk, gv = caches[s].read_rows(0, base + r, 1)
            assert np.array_equal(gk.reshape(-1), store(k[r]).reshape(-1)), (s, base, r)
            assert np.array_equal(gv.reshape(-1), store(v[r]).reshape(-1)), (s, base, r)
    pool.close()


# Blocks of several tiles, cut by the estimates: contexts left whole that the even fill had split (on four and eight
# wavefronts and on halves of blocks), fewer and more splits than it, another form at as many; contexts of one length,
# nearly so, and far apart (which keep the even fill). `splits` and `wavefronts` are the launch's on 256 compute units,
# the even fill's in the comment.
@pytest.mark.parametrize("elem,d,q_heads,kv_heads,rows,ctxs,splits,wavefronts", [
    ("f16", 192, 32, 4, 38, (198, 198, 198), 1, "4"),                  # 2, 4
    ("f16", 240, 8, 1, 33, (1206, 1190), 6, "4"),                      # 10, 4
    ("f16", 144, 8, 8, 25, (610,), 5, "4"),                            # the same
    ("f16", 80, 32, 4, 13, (911,) * 7, 1, "8"),                        # 2, 4
    ("f16", 48, 6, 2, 12, (507,), 1, "8"),                             # 5, 4
    ("f16", 112, 32, 4, 19, (346,), 1, "4"),                           # 1, 8
    ("f16", 112, 32, 4, 20, (1239,), 6, "4"),                          # 10, 4
    ("f16", 48, 6, 2, 9, (333, 320), 1, "8"), ("f16", 112, 32, 4, 9, (700, 90), 1, "8"),  # the same, far apart
    ("f32", 64, 32, 4, 12, (845, 840, 833, 845, 845, 845, 845, 831), 1, "8"),  # 2, 4
    ("f32", 64, 32, 4, 28, (1191,), 4, "8"),                           # 8, 4
    ("f32", 64, 24, 8, 3, (1500, 30), 24, "4,half_blocks"),            # the same, far apart
    ("f32", 128, 32, 4, 19, (635,) * 6, 1, "4,half_blocks"),           # 2, 4
    ("f32", 128, 8, 1, 25, (363, 345, 345, 345, 345), 7, "4,half_blocks"),  # 4, 4
    ("f32", 128, 32, 4, 25, (675, 642, 642, 642, 642), 3, "4"),        # 2, 4
    ("f32", 128, 32, 4, 21, (778, 778), 5, "4,half_blocks"),           # 5, 4
    ("f32", 128, 8, 1, 15, (1900, 1891), 15, "4"),                     # the same
    ("f32", 128, 32, 4, 3, (614,) * 7, 4, "4,half_blocks"),            # 5, 4
])
def test_blocks_of_several_tiles(elem, d, q_heads, kv_heads, rows, ctxs, splits, wavefronts, capfd):
    P = pkg()
    rng = np.random.default_rng(d + rows)
    pool = P.KvPool([P.LayerKind.Global], kv_heads, d, elem=elem, max_slots=len(ctxs), capacity_rows=max(ctxs) + rows + 8)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in ctxs]
    refs = [oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d, store_f16=elem == "f16") for _ in ctxs]
    for cache, ref, n in zip(caches, refs, ctxs):
        k, v = normal(rng, n, kv_heads * d), normal(rng, n, kv_heads * d)
        cache.restore_bulk(0, 0, k, v)
        ref.restore_bulk(0, 0, k, v)
    total = rows * len(ctxs)
    q, k, v = normal(rng, total, q_heads * d), normal(rng, total, kv_heads * d), normal(rng, total, kv_heads * d)
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = torch.full_like(qd, float("nan"))
    lib = P._native.load()
    capfd.readouterr()
    lib.itak_set_debug_enabled(1)
    try:
        pool.attention_step_device(0, [(c, rows) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
    finally:
        lib.itak_set_debug_enabled(0)
    torch.cuda.synchronize()
    said = dict(w.split("=", 1) for w in capfd.readouterr().err.split() if "=" in w)
    assert (int(said["splits"]), said["wavefronts"]) == (splits, wavefronts)
    got = out.cpu().numpy()
    for s, ref in enumerate(refs):
        at = slice(s * rows, (s + 1) * rows)
        want = oracle.attention_step(ref, 0, q[at], k[at], v[at], q_heads, ctxs[s], threads=8)
        assert rel_err(got[at].reshape(-1), want) <= 1e-5, s
    pool.close()
