"""Steps of many slots: every workgroup of the attention launch and of the merge finds the item it belongs to
among the batch's. Counts at the edges of the argument blocks (1, 8 and 64 items), slots of very different
lengths, so that the items' shares of both launches differ and some are left whole where others are split."""
import numpy as np
import pytest
import torch

import oracle
from helpers import max_abs, normal, pkg

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("slots", [2, 7, 8, 9, 63, 64, 65])
@pytest.mark.parametrize("elem,d", [("f16", 128), ("f32", 128), ("f16", 80), ("f16", 66)])
def test_every_workgroup_finds_its_item(elem, d, slots):
    P = pkg()
    rng = np.random.default_rng(1000 * slots + d)
    kvh, q_heads = 2, 8
    row = kvh * d
    contexts = [int(n) for n in rng.integers(1, 90, slots)]
    for at in (0, slots // 2, slots - 1):  # long ones at either end and between
        contexts[at] = int(rng.integers(600, 1100))
    rows = [int(r) for r in rng.choice([1, 1, 1, 2, 3], slots)]
    pool = P.KvPool([P.LayerKind.Global], kvh, d, elem=elem, max_slots=slots, capacity_rows=1112)
    pool.set_stream(torch.cuda.current_stream().cuda_stream)
    caches = [pool.acquire() for _ in range(slots)]
    refs = [oracle.KvCache.new([oracle.LayerKind.Global], kvh, d, store_f16=(elem == "f16")) for _ in range(slots)]
    for cache, ref, n in zip(caches, refs, contexts):
        k, v = normal(rng, n, row), normal(rng, n, row)
        kd, vd = dev(k), dev(v)
        pool.append_device(0, [(cache, n)], kd.data_ptr(), vd.data_ptr())
        torch.cuda.synchronize()
        for p in range(n):
            ref.append(0, k[p], v[p], p)
    for step_rows in ([1] * slots, rows):
        total = sum(step_rows)
        q, k, v = normal(rng, total, q_heads * d), normal(rng, total, row), normal(rng, total, row)
        qd, kd, vd = dev(q), dev(k), dev(v)
        out = torch.full_like(qd, float("nan"))
        pool.attention_step_device(0, list(zip(caches, step_rows)), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                   out.data_ptr(), q_heads)
        torch.cuda.synchronize()
        got, at = out.cpu().numpy(), 0
        for s, (ref, n) in enumerate(zip(refs, step_rows)):
            want = oracle.attention_step(ref, 0, q[at:at + n], k[at:at + n], v[at:at + n], q_heads, contexts[s])
            err = max_abs(got[at:at + n].reshape(-1), want)
            if elem == "f32":
                err /= float(np.abs(want).max())
            # (Of f16 pools only head_dim 128 rounds queries and weights to f16: the others' arithmetic is f32's.)
            bar = 1e-5 if elem == "f32" else 2e-3 if d == 128 else 5e-5
            assert err <= bar, (slots, s, n, contexts[s], err)
            at += n
            contexts[s] += n
    pool.close()
