"""The tiles kernel (f16 pools at head_dim 128: prompt chunks and speculative blocks whose rows are
cut in tiles of 16 or 32 query vectors, the wavefronts sharing out the keys) against the CPU oracle,
around its edges: tiles with a remainder, groups that do not divide 16, new rows that begin and end
anywhere in a block, as many new blocks as a launch brings along and more (appended before it), contexts
whole and split, causal and windowed tiles that see only part of a split's run, rings that wrap. The
oracle's f16 cache rounds keys and values as the pool does; queries and weights enter the products as
halves, hence the f16 bar of 2e-3 on outputs of order one."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg

pytestmark = pytest.mark.gpu

D = 128


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.fixture
def kernels(capfd):
    lib = pkg()._native.load()
    lib.itak_set_debug_enabled(1)
    capfd.readouterr()
    yield lambda: [w[7:] for w in capfd.readouterr().err.split() if w.startswith("kernel=")]
    lib.itak_set_debug_enabled(0)


def setup(ctxs, rows, kv_heads, window, seed):
    P = pkg()
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    rng = np.random.default_rng(seed)
    pool = P.KvPool([kind], kv_heads, D, elem="f16", max_slots=len(ctxs), capacity_rows=max(ctxs) + rows + 8,
                    ring_headroom=max(64, rows))
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in ctxs]
    refs = [oracle.KvCache.new([okind], kv_heads, D, store_f16=True) for _ in ctxs]
    for cache, ref, n in zip(caches, refs, ctxs):
        first = 0 if window is None else max(0, n - window)
        if n:
            k, v = normal(rng, n - first, kv_heads * D), normal(rng, n - first, kv_heads * D)
            cache.restore_bulk(0, first, k, v)
            ref.restore_bulk(0, first, k, v)
    return rng, pool, caches, refs


def step(pool, caches, rows, q, k, v, q_heads, softcap=0.0):
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = torch.full_like(qd, float("nan"))
    pool.attention_step_device(0, [(c, rows) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                               out.data_ptr(), q_heads, softcap=softcap)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("softcap", [0.0, 20.0])
@pytest.mark.parametrize("ctxs,rows,q_heads,kv_heads,window", [
    ([0], 9, 32, 4, None), ([0], 128, 8, 1, None), ([0], 33, 6, 2, None),       # nothing but new rows; four blocks of them
    ([31], 9, 32, 4, None), ([32], 65, 8, 8, None), ([95], 98, 16, 1, None),    # first new row last / first in its block
    ([127], 130, 32, 4, None), ([300], 300, 16, 4, None),                       # more new blocks than a launch brings along
    ([300], 17, 15, 1, None), ([1000], 61, 32, 4, None), ([2500], 24, 32, 8, None),   # whole, then split
    ([90], 7, 32, 4, None), ([300, 33, 5], 5, 32, 4, None), ([290], 8, 32, 4, None),  # steps of few rows
    ([700, 40, 0, 128], 20, 16, 4, None),                                       # items of different lengths
    ([500], 61, 32, 4, 200), ([2100], 40, 8, 2, 1500), ([64], 30, 8, 1, 33),    # windows; a ring of four blocks
    ([4000], 200, 8, 1, 2000), ([40, 600], 12, 32, 4, 96),
])
def test_against_the_oracle(kernels, ctxs, rows, q_heads, kv_heads, window, softcap):
    rng, pool, caches, refs = setup(ctxs, rows, kv_heads, window, rows * 7 + len(ctxs))
    kernels()
    n = rows * len(ctxs)
    q, k, v = (normal(rng, n, w * D) for w in (q_heads, kv_heads, kv_heads))
    got = step(pool, caches, rows, q, k, v, q_heads, softcap).reshape(len(ctxs), -1)
    assert kernels() == ["tiles_f16"]
    for i, ref in enumerate(refs):
        at = slice(i * rows, (i + 1) * rows)
        want = oracle.attention_step(ref, 0, q[at], k[at], v[at], q_heads, ctxs[i],
                                     oracle.AttentionParams(softcap=softcap), threads=8)
        assert max_abs(got[i], np.asarray(want).reshape(-1)) <= 2e-3
        if window is not None:  # (the raw planes below look at rings)
            continue
        _, gk, gv = caches[i].read_rows(0, ctxs[i], rows)
        assert np.array_equal(gk.reshape(rows, -1), oracle.f32_to_f16_array(k[at]))
        assert np.array_equal(gv.reshape(rows, -1), oracle.f32_to_f16_array(v[at]))
    pool.close()


# New rows of more blocks than a workgroup of eight (four) wavefronts stores, first and last block begun or full.
@pytest.mark.parametrize("ctxs,rows,q_heads,kv_heads", [
    ([500], 200, 32, 4), ([1005], 140, 16, 4), ([480], 256, 8, 4), ([511], 129, 32, 4), ([600, 37], 130, 16, 4),
    ([1], 65, 16, 2)])
def test_new_rows_of_many_blocks(kernels, ctxs, rows, q_heads, kv_heads):
    test_against_the_oracle(kernels, ctxs, rows, q_heads, kv_heads, None, 0.0)


# A softcap far from one: steps that the split-K kernel takes as well stay with it, whose queries do not carry
# 2 log2(e) / softcap into their rounding (a factor of 261 on queries of some hundreds at the smallest one here).
@pytest.mark.parametrize("softcap,kernel", [(2.0 ** -10, "splitk_f16"), (1.9, "splitk_f16"), (2.0, "tiles_f16"),
                                            (1024.0, "tiles_f16"), (1100.0, "splitk_f16")])
def test_steps_of_few_rows_with_a_softcap_far_from_one(kernels, softcap, kernel):
    ctx, rows, q_heads, kv_heads = 290, 8, 32, 4
    rng, pool, (cache,), (ref,) = setup([ctx], rows, kv_heads, None, 11)
    q, k, v = (normal(rng, rows, w * D) for w in (q_heads, kv_heads, kv_heads))
    if softcap < 1.0:
        q *= 100.0
    kernels()
    got = step(pool, [cache], rows, q, k, v, q_heads, softcap)
    assert kernels() == [kernel]
    want = oracle.attention_step(ref, 0, q, k, v, q_heads, ctx, oracle.AttentionParams(softcap=softcap), threads=8)
    assert max_abs(got.reshape(-1), np.asarray(want).reshape(-1)) <= 2e-3
    pool.close()


# Steps the split-K kernel takes as well: tiles for contexts of up to 16 blocks (8 from eight KV heads on), beyond them
# for one slot.
@pytest.mark.parametrize("slots,rows,ctx,q_heads,kv_heads,kernel", [
    (2, 3, 509, 32, 4, "tiles_f16"), (2, 3, 510, 32, 4, "splitk_f16"), (1, 3, 510, 32, 4, "tiles_f16"),
    (1, 5, 251, 32, 8, "tiles_f16"), (1, 5, 252, 32, 8, "splitk_f16"), (2, 5, 252, 32, 8, "splitk_f16"),
    (1, 5, 507, 32, 8, "splitk_f16"), (1, 5, 508, 32, 8, "tiles_f16"), (2, 5, 508, 32, 8, "splitk_f16")])
def test_steps_of_few_rows_by_blocks_and_slots(kernels, slots, rows, ctx, q_heads, kv_heads, kernel):
    rng, pool, caches, refs = setup([ctx] * slots, rows, kv_heads, None, ctx)
    q, k, v = (normal(rng, slots * rows, w * D) for w in (q_heads, kv_heads, kv_heads))
    kernels()
    got = step(pool, caches, rows, q, k, v, q_heads).reshape(slots, -1)
    assert kernels() == [kernel]
    for i, ref in enumerate(refs):
        at = slice(i * rows, (i + 1) * rows)
        want = oracle.attention_step(ref, 0, q[at], k[at], v[at], q_heads, ctx, threads=8)
        assert max_abs(got[i], np.asarray(want).reshape(-1)) <= 2e-3
    pool.close()


# Steps of slots with different numbers of rows: a chunk of 128 rows and more beside others goes to the block kernel
# unless the tiles are estimated to be well ahead; a short one, or a chunk alone, as before.
@pytest.mark.parametrize("rows,ctxs,kernel", [
    ([7] * 10 + [22, 244], [46] * 10 + [317, 67], "prefill_f16"), ([1] * 3 + [128], [500] * 3 + [1000], "tiles_f16"),
    ([1] * 5 + [61], [300, 0, 77, 1500, 20, 333], "tiles_f16"), ([244], [67], "tiles_f16"),
    ([11], [8553], "prefill_f16")])  # (a near tie: the tiles' estimate is 3 % ahead)
def test_slots_of_different_row_counts(kernels, rows, ctxs, kernel):
    q_heads, kv_heads = 32, 8
    P = pkg()
    rng = np.random.default_rng(len(rows))
    pool = P.KvPool(1, kv_heads, D, elem="f16", max_slots=len(rows), capacity_rows=max(ctxs) + max(rows))
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in rows]
    refs = [oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, D, store_f16=True) for _ in rows]
    for cache, ref, n in zip(caches, refs, ctxs):
        if n:
            k, v = normal(rng, n, kv_heads * D), normal(rng, n, kv_heads * D)
            cache.restore_bulk(0, 0, k, v)
            ref.restore_bulk(0, 0, k, v)
    q, k, v = (normal(rng, sum(rows), w * D) for w in (q_heads, kv_heads, kv_heads))
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = torch.full_like(qd, float("nan"))
    kernels()
    pool.attention_step_device(0, list(zip(caches, rows)), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
    torch.cuda.synchronize()
    assert kernels() == [kernel]
    got, first = out.cpu().numpy(), 0
    for cache, ref, n, ctx in zip(caches, refs, rows, ctxs):
        at = slice(first, first + n)
        first += n
        want = oracle.attention_step(ref, 0, q[at], k[at], v[at], q_heads, ctx, threads=8)
        assert max_abs(got[at].reshape(-1), np.asarray(want).reshape(-1)) <= 2e-3
        _, gk, gv = cache.read_rows(0, ctx, n)
        assert np.array_equal(gk.reshape(n, -1), oracle.f32_to_f16_array(k[at]))
        assert np.array_equal(gv.reshape(n, -1), oracle.f32_to_f16_array(v[at]))
    pool.close()


# Rings of one and two blocks, where two position blocks of a step are the same storage block: its old rows
# are read beside the new ones' stores, and each row is in one place only.
@pytest.mark.parametrize("ctx,rows,window,headroom", [(20, 20, 1, 31), (7, 30, 2, 30), (300, 31, 1, 31), (20, 40, 20, 40),
                                                      (95, 34, 30, 34), (1000, 61, 3, 61), (63, 9, 16, 40)])
def test_rings_of_one_and_two_blocks(kernels, ctx, rows, window, headroom):
    q_heads, kv_heads = 32, 4
    P = pkg()
    rng = np.random.default_rng(ctx)
    pool = P.KvPool([P.LayerKind.windowed(window)], kv_heads, D, elem="f16", capacity_rows=ctx + 3 * rows, ring_headroom=headroom)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    cache = pool.acquire()
    ref = oracle.KvCache.new([oracle.LayerKind.windowed(window)], kv_heads, D, store_f16=True)
    first = max(0, ctx - window)
    k, v = normal(rng, ctx - first, kv_heads * D), normal(rng, ctx - first, kv_heads * D)
    cache.restore_bulk(0, first, k, v)
    ref.restore_bulk(0, first, k, v)
    for at in (ctx, ctx + rows, ctx + 2 * rows):
        q, k, v = (normal(rng, rows, w * D) for w in (q_heads, kv_heads, kv_heads))
        kernels()
        got = step(pool, [cache], rows, q, k, v, q_heads)
        assert kernels() == ["tiles_f16"]
        want = oracle.attention_step(ref, 0, q, k, v, q_heads, at, threads=8)
        assert max_abs(got.reshape(-1), np.asarray(want).reshape(-1)) <= 2e-3
    pool.close()


# The stored planes, raw, are what the row kernel writes: no byte beside the new rows', NaNs canonical.
@pytest.mark.parametrize("ctx,rows,window", [(0, 61, None), (45, 61, None), (31, 9, None), (40, 61, 33), (333, 40, 64)])
def test_new_rows_are_stored_as_the_row_kernel_stores_them(kernels, ctx, rows, window):
    planes = []
    for appended_before in (True, False):
        rng, pool, (cache,), _ = setup([ctx], rows, 2, window, 5)
        q, k, v = (normal(rng, rows, w * D) for w in (8, 2, 2))
        k[1, 3], v[rows - 1, 5], v[2, 7], k[0, 9] = np.nan, np.inf, -np.nan, 1e30
        kernels()
        if appended_before:
            kd, vd = dev(k), dev(v)
            pool.append_device(0, [(cache, rows)], kd.data_ptr(), vd.data_ptr())
            torch.cuda.synchronize()
        else:
            step(pool, [cache], rows, q, k, v, 8)
            assert kernels() == ["tiles_f16"]
        planes.append(cache.read_raw(0))
        pool.close()
    for got, want in zip(*planes):
        assert np.array_equal(np.asarray(got).view(np.uint8), np.asarray(want).view(np.uint8))


# Values that are not finite reach exactly the rows that see them: a later row of the step, a ring
# row that only the first rows' windows hold, one that nobody sees.
@pytest.mark.parametrize("ctx,rows,window", [(333, 20, 96), (700, 61, None), (0, 40, None), (200, 7, None)])
def test_values_that_are_not_finite(kernels, ctx, rows, window):
    kv_heads, q_heads = 4, 32
    P = pkg()
    rng = np.random.default_rng(ctx + rows)
    k, v = normal(rng, ctx + rows, kv_heads * D), normal(rng, ctx + rows, kv_heads * D)
    q = normal(rng, rows, q_heads * D)
    v[ctx + rows - 1, 5], v[ctx + rows // 2, D + 9], v[ctx + rows // 2, 2 * D + 1] = np.inf, -np.inf, np.nan
    if window:
        v[ctx + 1 - window, 3], v[ctx + 2 - window, D + 4], v[ctx - window, 7] = np.inf, np.nan, -np.inf
    kind, okind = ((m.LayerKind.Global if window is None else m.LayerKind.windowed(window)) for m in (P, oracle))
    pool = P.KvPool([kind], kv_heads, D, elem="f16", capacity_rows=ctx + rows, ring_headroom=64)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    cache, ref = pool.acquire(), oracle.KvCache.new([okind], kv_heads, D, store_f16=True)
    kd, vd = dev(k), dev(v)
    for at in range(0, ctx, 40):
        pool.append_device(0, [(cache, min(40, ctx - at))], kd[at:].data_ptr(), vd[at:].data_ptr())
    first = max(0, ctx - window) if window else 0
    if ctx:
        ref.restore_bulk(0, first, k[first:ctx], v[first:ctx])
    kernels()
    got = step(pool, [cache], rows, q, k[ctx:], v[ctx:], q_heads).reshape(-1)
    assert kernels() == ["tiles_f16"]
    want = np.asarray(oracle.attention_step(ref, 0, q, k[ctx:], v[ctx:], q_heads, ctx, threads=8)).reshape(-1)
    fin = np.isfinite(want)
    assert fin.any() and not fin.all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert max_abs(got[fin], want[fin]) <= 2e-3
    pool.close()


# The gate: applied by the launch itself for a context left whole, by the merge for a split one.
@pytest.mark.parametrize("ctx", [200, 3000])
def test_gate(kernels, ctx):
    rows, q_heads, kv_heads = 20, 32, 4
    rng, pool, (cache,), (ref,) = setup([ctx], rows, kv_heads, None, ctx)
    q, k, v, g = (normal(rng, rows, w * D) for w in (q_heads, kv_heads, kv_heads, q_heads))
    qd, kd, vd, gd = dev(q), dev(k), dev(v), dev(g)
    out = torch.full_like(qd, float("nan"))
    kernels()
    pool.attention_prep_step_device(0, [(cache, rows)], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(),
                                    q_heads, gate_ptr=gd.data_ptr())
    torch.cuda.synchronize()
    assert kernels() == ["tiles_f16"]
    want = oracle.attn_gate(oracle.attention_step(ref, 0, q, k, v, q_heads, ctx, threads=8), g)
    assert max_abs(out.cpu().numpy().reshape(-1), np.asarray(want).reshape(-1)) <= 2e-3
    pool.close()


# Rows that are stored already, asked by position: the newest `rows` positions, nothing brought along.
def test_rows_that_are_stored_already(kernels):
    ctx, rows, q_heads, kv_heads = 500, 30, 16, 4
    rng, pool, (cache,), (ref,) = setup([ctx], rows, kv_heads, None, 9)
    q = normal(rng, rows, q_heads * D)
    qd = dev(q)
    out = torch.full_like(qd, float("nan"))
    kernels()
    pool.attention_device(0, [(cache, rows)], qd.data_ptr(), out.data_ptr(), q_heads)
    torch.cuda.synchronize()
    assert kernels() == ["tiles_f16"]
    want = oracle.gqa_attention(q, rows, q_heads, list(range(ctx - rows, ctx)), ref.view(0), oracle.AttentionParams())
    assert max_abs(out.cpu().numpy().reshape(-1), np.asarray(want).reshape(-1)) <= 2e-3
    pool.close()
