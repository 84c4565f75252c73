"""One-row steps at head_dim 128 over contexts short enough to stay whole: every workgroup works out all scores of a
(slot, KV head) and a part of its channels, eight wavefronts taking a 32-key block each a round. Block counts at the
edges of the rounds, the new row at the edges of its block, groups and head counts that leave the deal of parts uneven,
slots of unequal lengths (eight, four and two parts), layers with a window before and after its ring has wrapped.

The bar against the oracle over the same f16 rows: rounding a query and a weight to f16 is 2^-11 of either at most. A score's
128 terms, of size 0.64^2 / 11.3 each on normal rows, are off by 2^-12 of their size on average and either sign, so it is off by 2^-12 * 128^.5 *
0.1 = 3e-4, and an output, a mean of |v| <= 4 with those weights, by less than 4 * (3e-4 + 2^-12) = 2e-3. Rows
stored are exact."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg

pytestmark = pytest.mark.gpu

D = 128


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("q_heads,kv_heads,slots", [(32, 4, 1), (8, 8, 1), (32, 2, 3), (27, 9, 4), (5, 1, 8), (32, 4, 17)])
@pytest.mark.parametrize("window", [None, 100, 512])
def test_short_steps_by_channels(q_heads, kv_heads, slots, window):
    P = pkg()
    row = kv_heads * D
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    for n in (0, 1, 31, 32, 255, 256, 511, 512, 767, 768):
        rng = np.random.default_rng(n + 1000 * slots)
        pool = P.KvPool([kind], kv_heads, D, elem="f16", max_slots=slots, capacity_rows=800)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        caches, refs, lengths = [], [], []
        for s in range(slots):
            length = max(n - 37 * s, 0)
            first = 0 if window is None else max(0, length - window)
            cache, ref = pool.acquire(), oracle.KvCache.new([okind], kv_heads, D, store_f16=True)
            if length:
                k, v = normal(rng, length - first, row), normal(rng, length - first, row)
                cache.restore_bulk(0, first, k, v)
                ref.restore_bulk(0, first, k, v)
            caches.append(cache), refs.append(ref), lengths.append(length)
        for step in range(2):
            q, k, v = normal(rng, slots, q_heads * D), normal(rng, slots, row), normal(rng, slots, row)
            qd, kd, vd = dev(q), dev(k), dev(v)
            out = torch.full_like(qd, float("nan"))
            softcap = 30.0 * step
            pool.attention_step_device(0, [(c, 1) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                       out.data_ptr(), q_heads, softcap=softcap)
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            for s, ref in enumerate(refs):
                at = lengths[s] + step
                want = oracle.attention_step(ref, 0, q[s:s + 1], k[s:s + 1], v[s:s + 1], q_heads, at,
                                             oracle.AttentionParams(softcap=softcap))
                assert max_abs(got[s], want) <= 2e-3, (n, s, at, max_abs(got[s], want))
                _, gk, gv = caches[s].read_rows(0, caches[s].stored_len(0) - 1, 1)
                assert np.array_equal(gk.reshape(-1), oracle.f32_to_f16_array(k[s]))
                assert np.array_equal(gv.reshape(-1), oracle.f32_to_f16_array(v[s]))
        pool.close()


@pytest.mark.parametrize("q_heads,kv_heads,slots", [(32, 4, 1), (32, 2, 3), (27, 9, 4), (32, 4, 9), (10, 5, 14)])
@pytest.mark.parametrize("window", [None, 100, 512])
def test_short_preparing_steps_by_channels(q_heads, kv_heads, slots, window):
    from test_gpu_prep import run_case

    for i, n in enumerate((0, 1, 31, 32, 255, 256, 383, 440, 500, 580)):
        run_case("f16", q_heads, kv_heads, D, n, 1, norm=True, rope_base=(1e4, 0.0, 5e5)[i % 3],
                 interleaved=bool(i & 1), rotary=(0, 64)[i % 2], gate=i % 4 != 2, seed=n, slots=slots, window=window)


# Other head dims on blocked f16 planes: queries and weights as three halves, so the bar is what f32 sums of a thousand
# terms leave, 2^-23 * 1024 of |v| <= 4 at most and a tenth of that as they are of either sign: 5e-5. Every count of
# channel tiles, parts of one tile and of several (the last of which may be part empty), one to four rounds, and runs of
# eight blocks merged by a second launch, of slots whole beside split ones; `bad` plants an infinity in a stored key and value and in the
# new row, whose rows then are the oracle's, infinities and NaN as they are.
@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("d,q_heads,kv_heads,slots", [(16, 8, 2, 1), (32, 8, 8, 2), (64, 32, 4, 1), (64, 16, 1, 9), (80, 32, 8, 1),
                                                      (80, 9, 3, 10), (96, 32, 4, 3), (112, 14, 2, 1), (112, 32, 4, 8), (144, 8, 4, 1),
                                                      (192, 32, 4, 1), (208, 8, 8, 3), (256, 32, 4, 1), (256, 16, 2, 12), (80, 32, 8, 5), (112, 8, 8, 6)])
@pytest.mark.parametrize("window", [None, 100])
def test_short_steps_at_other_head_dims(d, q_heads, kv_heads, slots, window, bad):
    P = pkg()
    row = kv_heads * d
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    for n in (0, 31, 32, 255, 256, 511, 767, 800, 1023, 1056):
        rng = np.random.default_rng(n + 1000 * slots + d)
        pool = P.KvPool([kind], kv_heads, d, elem="f16", max_slots=slots, capacity_rows=1060)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        caches, refs, lengths = [], [], []
        for s in range(slots):
            length = max(n - 37 * s, 0)
            first = 0 if window is None else max(0, length - window)
            cache, ref = pool.acquire(), oracle.KvCache.new([okind], kv_heads, d, store_f16=True)
            if length:
                k, v = normal(rng, length - first, row), normal(rng, length - first, row)
                if bad:
                    v[rng.integers(length - first), rng.integers(row)] = np.inf
                    k[rng.integers(length - first), rng.integers(row)] = -np.inf
                cache.restore_bulk(0, first, k, v)
                ref.restore_bulk(0, first, k, v)
            caches.append(cache), refs.append(ref), lengths.append(length)
        for step in range(2):
            q, k, v = normal(rng, slots, q_heads * d), normal(rng, slots, row), normal(rng, slots, row)
            if bad:
                v[0, rng.integers(row)] = -np.inf
            qd, kd, vd = dev(q), dev(k), dev(v)
            out = torch.full_like(qd, 7.0)
            softcap = 30.0 * step
            pool.attention_step_device(0, [(c, 1) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                       out.data_ptr(), q_heads, softcap=softcap)
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            for s, ref in enumerate(refs):
                at = lengths[s] + step
                want = np.asarray(oracle.attention_step(ref, 0, q[s:s + 1], k[s:s + 1], v[s:s + 1], q_heads, at,
                                                        oracle.AttentionParams(softcap=softcap))).reshape(-1)
                finite = np.isfinite(want)
                assert np.array_equal(got[s][~finite], want[~finite], equal_nan=True), (n, s, at)
                assert not finite.any() or max_abs(got[s][finite], want[finite]) <= 5e-5, (n, s, at)
                _, gk, gv = caches[s].read_rows(0, caches[s].stored_len(0) - 1, 1)
                assert np.array_equal(gk.reshape(-1), oracle.f32_to_f16_array(k[s]))
                assert np.array_equal(gv.reshape(-1), oracle.f32_to_f16_array(v[s]))
        pool.close()


# Contexts cut into runs of fewer than eight blocks, so that some wavefronts of a workgroup have none: 33 and 34 blocks are five
# runs of seven and a rest, 41 six, 9 beside them two of five. Keys that are large in one channel of every row, as a
# bias on their projection leaves them, or in the first eight, with queries of one sign: a score made up from a part of a row is far
# from every true one.
#
# The bar: a score is a sum of d terms, and f32 leaves it off by 2^-24 * d^.5 of the sum of their sizes; an output, a mean of
# |v| <= 4, by as much of 4 on either side of the comparison, beside the 5e-5 above.
@pytest.mark.parametrize("contexts", [(1040,), (1060,), (1300,), (1300, 270), (270, 1060, 1040)])
@pytest.mark.parametrize("d,q_heads,kv_heads", [(64, 32, 4), (80, 32, 4), (112, 14, 2), (256, 32, 4), (256, 8, 2)])
@pytest.mark.parametrize("keys", ["a bias on one channel", "eight large channels"])
def test_runs_of_fewer_blocks_than_wavefronts(d, q_heads, kv_heads, contexts, keys):
    P = pkg()
    row, slots, group = kv_heads * d, len(contexts), q_heads // kv_heads
    rng = np.random.default_rng(d + sum(contexts))
    bias = np.zeros((kv_heads, d), np.float32)
    if keys == "eight large channels":
        bias[:, :8] = 4.5
    else:
        for h in range(kv_heads):
            bias[h, rng.integers(8)] = rng.choice([-1, 1]) * rng.integers(150, 400)
    def some_keys(n):
        return 0.25 * normal(rng, n, row) + bias.reshape(1, row)
    pool = P.KvPool([P.LayerKind.Global], kv_heads, d, elem="f16", max_slots=slots, capacity_rows=1320)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches, refs, stored = [], [], []
    for length in contexts:
        cache, ref = pool.acquire(), oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d, store_f16=True)
        k, v = some_keys(length), normal(rng, length, row)
        cache.restore_bulk(0, 0, k, v)
        ref.restore_bulk(0, 0, k, v)
        caches.append(cache), refs.append(ref), stored.append(np.abs(k).reshape(length, kv_heads, d).max(0))
    q = 2 * normal(rng, slots, q_heads * d) if keys == "a bias on one channel" else 4 + 0.5 * normal(rng, slots, q_heads * d)
    k, v = some_keys(slots), normal(rng, slots, row)
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = torch.full_like(qd, float("nan"))
    pool.attention_step_device(0, [(c, 1) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for s, ref in enumerate(refs):
        want = oracle.attention_step(ref, 0, q[s:s + 1], k[s:s + 1], v[s:s + 1], q_heads, contexts[s])
        most = np.maximum(stored[s], np.abs(k[s]).reshape(kv_heads, d)).repeat(group, 0)
        size = float((np.abs(q[s]).reshape(q_heads, d) * most).sum(1).max()) / d ** 0.5
        bar = 5e-5 + 2 * 4 * size * 2.0 ** -24 * d ** 0.5
        assert max_abs(got[s], want) <= bar, (s, contexts[s], max_abs(got[s], want), bar)
    pool.close()


@pytest.fixture
def launches(capfd):
    """(kernel, wavefronts) of the attention launches since the last look, from the diagnostic channel."""
    lib = pkg()._native.load()
    lib.itak_set_debug_enabled(1)
    capfd.readouterr()

    def since():
        words = [w.split("=", 1) for w in capfd.readouterr().err.split()]
        return list(zip([w[1] for w in words if w[0] == "kernel"], [w[1] for w in words if w[0] == "wavefronts"]))
    yield since
    lib.itak_set_debug_enabled(0)


# The lines of the two planners on a device of 256 compute units: which kernel a step goes to and how it is cut there.
@pytest.mark.parametrize("d,q_heads,kv_heads,slots,n,form,kernel,wavefronts", [
    (128, 32, 4, 1, 0, {}, "whole_f16", "8,parts=8"), (128, 32, 4, 1, 639, {}, "whole_f16", "8,parts=8"),
    (128, 32, 4, 1, 640, {}, "splitk_f16", "-"), (128, 32, 4, 8, 767, {}, "whole_f16", "8,parts=8"),
    (128, 32, 4, 8, 768, {}, "splitk_f16", "-"), (128, 32, 4, 9, 500, {}, "whole_f16", "8,parts=4"),
    (128, 32, 4, 16, 767, {}, "whole_f16", "8,parts=4"), (128, 32, 4, 17, 500, {}, "whole_f16", "8,parts=2"),
    (128, 32, 4, 24, 500, {}, "whole_f16", "8,parts=2"), (128, 32, 4, 25, 500, {}, "splitk_f16", "-"),
    (128, 8, 8, 1, 95, {}, "whole_f16", "8,parts=8"), (128, 8, 8, 1, 96, {}, "splitk_f16", "-"), (128, 2, 1, 1, 127, {}, "splitk_f16", "-"),
    (128, 8, 8, 1, 128, {}, "whole_f16", "8,parts=8"), (128, 3, 1, 1, 127, {}, "whole_f16", "8,parts=8"),
    (128, 32, 4, 8, 127, {}, "whole_f16", "8,parts=8"), (128, 32, 4, 9, 127, {}, "splitk_f16", "-"),
    (128, 32, 4, 9, 128, {}, "whole_f16", "8,parts=4"), (128, 8, 8, 1, 127, {"prep": True}, "whole_f16", "8,parts=8"),
    (128, 8, 8, 2, 127, {"prep": True}, "splitk_f16", "-"),
    (128, 32, 1, 1, 300, {}, "splitk_f16", "-"), (128, 32, 4, 1, 300, {"merge_in_launch": True}, "splitk_f16", "-"),
    (128, 32, 4, 1, 300, {"q_two_halves": True}, "splitk_f16", "-"), (128, 32, 4, 1, 300, {"die_merge": True}, "splitk_f16", "-"),
    (128, 32, 4, 1, 383, {"prep": True}, "whole_f16", "8,parts=8"), (128, 32, 4, 1, 384, {"prep": True}, "splitk_f16", "-"),
    (64, 32, 4, 1, 767, {}, "parts_halves", "8,tiles=1"), (80, 32, 8, 1, 800, {}, "parts_halves", "8,tiles=1"),
    (80, 32, 8, 6, 700, {}, "parts_halves", "8,tiles=1"), (80, 32, 8, 8, 700, {}, "parts_halves", "8,tiles=2"),
    (80, 32, 8, 8, 1500, {}, "splitk_any", "4"), (256, 32, 4, 1, 511, {}, "parts_halves", "8,tiles=2"),
    (256, 32, 4, 1, 1500, {}, "parts_halves", "8,tiles=2"), (256, 32, 4, 4, 1500, {}, "parts_halves", "8,tiles=8")])
def test_which_steps_go_by_channels(launches, d, q_heads, kv_heads, slots, n, form, kernel, wavefronts):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are counted in compute units")
    form = dict(form)
    prep = form.pop("prep", False)
    pool = pkg().KvPool(1, kv_heads, d, elem="f16", max_slots=slots, capacity_rows=n + 1,
                        **{"q_two_halves": False, "die_merge": False, **form})
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    items = [(pool.acquire(), 1) for _ in range(slots)]
    rows = torch.ones(max(slots * n, 1), kv_heads * d, device="cuda")
    if n:
        pool.append_device(0, [(c, n) for c, _ in items], rows.data_ptr(), rows.data_ptr())
    q, k = torch.ones(slots, q_heads * d, device="cuda"), torch.ones(slots, kv_heads * d, device="cuda")
    out = torch.zeros_like(q)
    launches()
    step = pool.attention_prep_step_device if prep else pool.attention_step_device
    step(0, items, q.data_ptr(), k.data_ptr(), k.data_ptr(), out.data_ptr(), q_heads)
    torch.cuda.synchronize()
    assert launches() == [(kernel, wavefronts)]
    assert torch.allclose(out, torch.ones_like(out), atol=1e-3)  # every value row is ones
    pool.close()


# Outputs over the queries, or over the new rows where there are as many heads of either: steps by channels, whose workgroups would
# read what others have written over, leave them to the forms that took them before. Memory that only adjoins is no such case.
# Bars as above.
IN_PLACE = [(128, 32, 4, (300,)), (128, 8, 8, (90, 700, 31)), (128, 16, 4, (500,) * 17), (64, 16, 16, (400,)), (80, 32, 8, (400, 90)),
            (256, 8, 8, (300,)), (112, 14, 2, (1300, 200))]


@pytest.mark.parametrize("d,heads,kv_heads,contexts,over", [
    (*shape, over) for shape in IN_PLACE for over in ("q", "k", "v", "nothing") if over not in "kv" or shape[1] == shape[2]])
@pytest.mark.parametrize("form", ["step", "preparing", "allocation-free"])
def test_outputs_over_the_inputs(launches, d, heads, kv_heads, contexts, over, form):
    P = pkg()
    rng = np.random.default_rng(d + sum(contexts))
    row, slots = kv_heads * d, len(contexts)
    pool = P.KvPool(1, kv_heads, d, elem="f16", max_slots=slots, capacity_rows=1400, q_two_halves=False, die_merge=False)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches, refs = [], []
    for length in contexts:
        cache, ref = pool.acquire(), oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, d, store_f16=True)
        k, v = normal(rng, length, row), normal(rng, length, row)
        cache.restore_bulk(0, 0, k, v)
        ref.restore_bulk(0, 0, k, v)
        caches.append(cache), refs.append(ref)
    q, k, v = normal(rng, slots, heads * d), normal(rng, slots, row), normal(rng, slots, row)
    memory = torch.from_numpy(np.concatenate([q.ravel(), k.ravel(), v.ravel(), np.zeros(q.size, np.float32)])).cuda()
    at, size = {}, {"q": q.size, "k": k.size, "v": v.size, "nothing": q.size}
    first = 0
    for name, n in size.items():
        at[name] = memory[first:first + n]
        first += n
    step = {"step": pool.attention_step_device, "preparing": pool.attention_prep_step_device,
            "allocation-free": pool.attention_step_device_noalloc}[form]
    launches()
    step(0, [(c, 1) for c in caches], at["q"].data_ptr(), at["k"].data_ptr(), at["v"].data_ptr(), at[over].data_ptr(), heads)
    torch.cuda.synchronize()
    by_channels, other = ("whole_f16", "splitk_f16") if d == 128 else ("parts_halves", "splitk_any")
    # (Prepared queries and keys of the other head dims are the pool's own memory, and preparing steps stay whole up to 12 blocks.)
    apart = over == "nothing" or (form == "preparing" and d != 128 and over != "v")
    if form != "preparing" or d != 128 or max(contexts) < 384:
        assert [kernel for kernel, _ in launches()] == [by_channels if apart else other]
    got = at[over].cpu().numpy().reshape(slots, -1)
    for s, ref in enumerate(refs):
        want = oracle.attention_step(ref, 0, q[s:s + 1], k[s:s + 1], v[s:s + 1], heads, contexts[s])
        assert max_abs(got[s], want) <= (2e-3 if d == 128 else 5e-5), (s, max_abs(got[s], want))
        for rows, new in zip(caches[s].read_rows(0, contexts[s], 1)[1:], (k, v)):
            assert np.array_equal(rows.reshape(-1), oracle.f32_to_f16_array(new[s]))
    pool.close()


# Queries near the ends of f16's range: what is rounded to f16 is the query or the query with the scale on, by the step's blocks
# (a batch's longest counts), and channels that fit in one of the two alone must find it. `most`: the largest channel.
#
# The bar: rounding moves a score by 2^-11 of its largest term at most, here of `term`, and a weight by 2^-11 of itself, so an
# output, a mean of |v| <= 5, by 2 * 5 * 2^-11 * (term + 1).
@pytest.mark.parametrize("contexts,q_heads,kv_heads,scale,most", [
    ((60,), 32, 4, 1.0, 6e4), ((127,), 32, 4, 1.0, 6e4), ((384,), 32, 4, 1.0, 6e4), ((639,), 16, 4, 1.0, 6e4),  # as they are
    ((767, 30) * 6, 8, 4, 1.0, 6e4), ((520,) * 15, 32, 4, 1.0, 6e4),
    ((128,), 32, 4, None, 4e5), ((383,), 32, 4, None, 4e5), ((90, 200), 16, 4, None, 4e5),                      # with the scale on
    ((60, 700) * 8, 8, 4, None, 4e5), ((300,) * 17, 8, 4, None, 4e5)])
def test_queries_at_the_ends_of_f16(launches, contexts, q_heads, kv_heads, scale, most):
    P = pkg()
    rng = np.random.default_rng(sum(contexts))
    row, slots, term = kv_heads * D, len(contexts), 0.5
    pool = P.KvPool(1, kv_heads, D, elem="f16", max_slots=slots, capacity_rows=800, q_two_halves=False, die_merge=False)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    at = scale or D ** -0.5
    large = rng.integers(D)

    def some_keys(n):
        k = 0.01 * normal(rng, n, row).reshape(n, kv_heads, D)
        k[:, :, large] = rng.uniform(-term, term, (n, kv_heads)) / (most * at)
        return k.reshape(n, row)
    q = normal(rng, slots, q_heads * D)
    q.reshape(slots, q_heads, D)[:, :, large] = rng.choice([-1, 1], (slots, q_heads)) * rng.uniform(0.9, 1, (slots, q_heads)) * most
    caches, refs = [], []
    for length in contexts:
        cache, ref = pool.acquire(), oracle.KvCache.new([oracle.LayerKind.Global], kv_heads, D, store_f16=True)
        k, v = some_keys(length), normal(rng, length, row)
        cache.restore_bulk(0, 0, k, v)
        ref.restore_bulk(0, 0, k, v)
        caches.append(cache), refs.append(ref)
    k, v = some_keys(slots), normal(rng, slots, row)
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = torch.full_like(qd, float("nan"))
    launches()
    pool.attention_step_device(0, [(c, 1) for c in caches], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads,
                               scale=scale)
    torch.cuda.synchronize()
    assert [kernel for kernel, _ in launches()] == ["whole_f16"]
    got = out.cpu().numpy()
    for s, ref in enumerate(refs):
        want = oracle.attention_step(ref, 0, q[s:s + 1], k[s:s + 1], v[s:s + 1], q_heads, contexts[s],
                                     oracle.AttentionParams(scale=scale))
        assert max_abs(got[s], want) <= 2 * 5 * 2.0 ** -11 * (term + 1), (s, max_abs(got[s], want))
    pool.close()
