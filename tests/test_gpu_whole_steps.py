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
