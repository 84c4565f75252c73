"""Steps longer than a windowed layer's window, cut back afterwards: every row the step brought is in
the ring, those below the window of its last row among them, because a cut of up to the ring's headroom
brings them into view again (the reference keeps what a rewind needs, crates/attention/src/cache.rs:
678-697). Rows bit for bit; the step's output, and that of the next step over the rows that were cut
back to, within the bars of the element type (f32 1e-5 relative, f16 2e-3 max-abs)."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elem,d,q_heads,kv_heads,window,headroom,held,rows,drop", [
    ("f32", 128, 8, 1, 128, 200, 0, 200, 100),    # 100 tiles of 16 vectors; the last sees rows 72 ..
    ("f32", 64, 8, 1, 128, 200, 37, 200, 100),
    ("f32", 96, 8, 1, 128, 200, 0, 200, 100),
    ("f32", 20, 3, 3, 16, 150, 70, 140, 129),     # one query head a KV head: a tile is 16 rows
    ("f32", 64, 6, 2, 50, 120, 33, 120, 117),     # a group of three: tiles begin inside a row
    ("f32", 128, 16, 1, 512, 1024, 0, 1024, 2),   # a chunk of two windows, two positions dropped
    ("f32", 128, 40, 1, 24, 70, 90, 70, 70),      # more than 16 query heads a KV head, all dropped
    ("f16", 128, 32, 4, 3, 64, 40, 8, 7),         # the launches that carry a few f16 rows
    ("f16", 80, 32, 4, 3, 64, 40, 8, 7),
    ("f16", 100, 16, 2, 3, 64, 29, 8, 8),
    ("f16", 128, 8, 1, 20, 64, 25, 60, 55),
    ("f16", 64, 8, 1, 20, 64, 25, 60, 55),
])
def test_a_cut_after_a_step_longer_than_the_window(elem, d, q_heads, kv_heads, window, headroom, held, rows, drop):
    rng = np.random.default_rng(d * 1000 + rows)
    width, f16 = kv_heads * d, elem == "f16"
    pool = pkg().KvPool([pkg().LayerKind.windowed(window)], kv_heads, d, elem=elem, ring_headroom=headroom)
    cache = pool.acquire()
    kept, more = held + rows - drop, 5
    q, k, v = (normal(rng, held + rows + more, w) for w in (q_heads * d, width, width))

    def reference(n):  # a cache that was given the first n positions
        ref = oracle.KvCache.new([oracle.LayerKind.windowed(window)], kv_heads, d, store_f16=f16)
        for p in range(n):
            ref.append(0, k[p], v[p], p)
        return ref

    def step(first, n, qkv):
        qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in qkv)
        out = torch.full_like(qd, float("nan"))
        pool.attention_step_device(0, [(cache, n)], qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q_heads)
        pool.synchronize()
        want = oracle.attention_step(reference(first), 0, *qkv, q_heads, first, oracle.AttentionParams(), threads=8)
        got = out.cpu().numpy().reshape(-1)
        assert (max_abs(got, want) <= 2e-3) if f16 else (rel_err(got, want) <= 1e-5), first

    def same_rows(n):
        for got, want in zip(cache.view(0).rows()[1:], reference(n).view(0).rows()[1:]):
            want = oracle.f32_to_f16_array(want) if f16 else np.asarray(want)
            assert np.asarray(got).tobytes() == want.tobytes(), n

    for first in range(0, held, 32):
        n = min(32, held - first)
        kd, vd = torch.from_numpy(k[first:first + n]).cuda(), torch.from_numpy(v[first:first + n]).cuda()
        pool.append_device(0, [(cache, n)], kd.data_ptr(), vd.data_ptr())
        pool.synchronize()
    step(held, rows, (q[held:held + rows], k[held:held + rows], v[held:held + rows]))
    same_rows(held + rows)
    pool.truncate([cache], [kept])
    same_rows(kept)
    # The positions that were dropped come again, with other rows.
    for t in (k, v):
        t[kept:kept + more] = normal(rng, more, width)
    step(kept, more, (q[:more], k[kept:kept + more], v[kept:kept + more]))
    same_rows(kept + more)
    pool.close()
