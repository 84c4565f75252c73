"""Steps of several rows as 16-vector tiles (f16 pools at head_dim 128): groups that straddle tiles, last
tiles of one vector, contexts left whole on four and eight wavefronts, split ones, and batches whose items
have different numbers of tiles, against the CPU oracle; and a value that is not finite in a row that only
the last query row sees."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("window", [None, 200])
@pytest.mark.parametrize("q_heads,kv_heads", [(32, 4), (15, 3), (16, 1), (6, 6), (24, 8)])
@pytest.mark.parametrize("contexts", [(0, 90), (60, 3), (250, 140), (500, 31), (1500, 40), (1500, 1400)])
def test_tiled_steps(contexts, q_heads, kv_heads, window):
    P = pkg()
    d = 128
    most = min(8, 64 // (q_heads // kv_heads))
    kind = P.LayerKind.Global if window is None else P.LayerKind.windowed(window)
    okind = oracle.LayerKind.Global if window is None else oracle.LayerKind.windowed(window)
    rng = np.random.default_rng(sum(contexts) + q_heads)
    pool = P.KvPool([kind], kv_heads, d, elem="f16", max_slots=2, capacity_rows=1600)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in contexts]
    refs = [oracle.KvCache.new([okind], kv_heads, d, store_f16=True) for _ in contexts]
    for cache, ref, n in zip(caches, refs, contexts):
        k, v = normal(rng, n, kv_heads * d), normal(rng, n, kv_heads * d)
        if n:
            kd, vd = dev(k), dev(v)
        for at in range(0, n, 50):
            pool.append_device(0, [(cache, min(50, n - at))], kd[at:].data_ptr(), vd[at:].data_ptr())
        for i in range(n):
            ref.append(0, k[i], v[i], i)
    for i, rows in enumerate(((most, 1), (3, most - 1), (1, 2), (most, most))):
        total = sum(rows)
        q = normal(rng, total, q_heads * d)
        k, v = normal(rng, total, kv_heads * d), normal(rng, total, kv_heads * d)
        if i == 3:
            v[rows[0] - 1, 5] = np.inf  # seen by the first item's last row alone
        qd, kd, vd = dev(q), dev(k), dev(v)
        out = torch.empty_like(qd)
        pool.attention_step_device(0, list(zip(caches, rows)), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                   out.data_ptr(), q_heads, softcap=30.0 if i == 1 else 0.0)
        torch.cuda.synchronize()
        got, at = out.cpu().numpy(), 0
        for s, r in enumerate(rows):
            want = np.asarray(oracle.attention_step(refs[s], 0, q[at:at + r], k[at:at + r], v[at:at + r], q_heads,
                                                    refs[s].next_position(0),
                                                    oracle.AttentionParams(softcap=30.0 if i == 1 else 0.0), threads=8)).reshape(-1)
            mine = got[at:at + r].reshape(-1)
            fine = np.isfinite(want)
            assert np.array_equal(np.isfinite(mine), fine) and (i == 3 and s == 0) == (not fine.all())
            assert max_abs(mine[fine], want[fine]) <= 2e-3, (rows, s)
            at += r
    pool.close()
