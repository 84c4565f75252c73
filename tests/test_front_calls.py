"""The per-layer calls of the Python front end, made by its compiled module for plain arguments and through ctypes
for every other kind: both make the same call."""
import warnings

import numpy as np
import pytest
import torch

from helpers import normal, pkg

gpu = pytest.mark.gpu


class Indexed:
    """A sequence that is neither a list nor a tuple."""

    def __init__(self, values):
        self._values = values

    def __len__(self):
        return len(self._values)

    def __iter__(self):
        return iter(self._values)


def front():
    hip = pkg().hip_compute
    hip._load()
    return hip._front


def test_only_plain_arguments_are_taken():
    f = front()
    items, ptrs = [(0, 1)], (1, 2, 3, 4)
    refused = 17  # InvalidArgument: no pool
    assert f.step(0, 0, items, *ptrs, 8, None, 0.0) == refused
    assert f.step(0, 0, tuple(items), *ptrs, 8, 0.5, 0) == refused
    for odd in ([(np.int64(0), 1)], [(0, np.uint32(1))], [[0, 1]], [(0, -1)], [(0, 1 << 32)], [(1 << 32, 1)], [(True, 1)],
                Indexed(items), items * 65):
        assert f.step(0, 0, odd, *ptrs, 8, None, 0.0) == -1
    for at in range(3, 8):
        args = [0, 0, items, *ptrs, 8, None, 0.0]
        args[at] = np.int64(1)
        assert f.step(*args) == -1
    assert f.step(0, 0, items, *ptrs, 8, np.float32(1), 0.0) == -1
    assert f.step(0, 0, items, *ptrs, 8, None, 10 ** 400) == -1
    assert f.truncate(0, [0], [5]) == refused
    assert f.truncate(0, [0], np.array([5])) == f.truncate(0, [0], [5, 6]) == f.truncate(0, [0], [-1]) == f.truncate(0, [0], [1 << 64]) == -1
    x = np.zeros((2, 8), np.float32)
    assert f.compute(0, 0, 0, x, x, x, 1, 0, 0.0, 1e4) == f.gqa(0, 0, 0, x, 2, 1, [0, 1], None, 0.0) == refused
    for odd in (x.astype(np.float64), x[:, ::2], x.astype(">f4"), x.tolist(), None):
        assert f.compute(0, 0, 0, odd, x, x, 1, 0, 0.0, 1e4) == f.gqa(0, 0, 0, odd, 2, 1, [0, 1], None, 0.0) == -1
    assert f.gqa(0, 0, 0, x, 2, 1, np.array([0, 1]), None, 0.0) == -1
    with pytest.raises(TypeError):
        f.step(0, 0, items)



# A library without its front module, or with one that is not this interpreter's, makes every call through ctypes and says so once.
@pytest.mark.parametrize("there", [None, b"", b"\x7fELF not a module"])
def test_a_library_without_its_front_module(monkeypatch, tmp_path, there):
    P = pkg()
    path = tmp_path / "front.so"
    if there is not None:
        path.write_bytes(there)
    monkeypatch.setattr(P._native, "FRONT_PATH", str(path))
    monkeypatch.setattr(P.hip_compute, "_front", None)
    with pytest.warns(RuntimeWarning, match="go through ctypes"):
        assert P.hip_compute._load() is P._native.load()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        f = front()  # (said once)
    x = np.zeros((2, 8), np.float32)
    assert f.step(0, 0, [(0, 1)], 1, 2, 3, 4, 8, None, 0.0) == f.truncate(0, [0], [5]) == -1
    assert f.compute(0, 0, 0, x, x, x, 1, 0, 0.0, 1e4) == f.gqa(0, 0, 0, x, 2, 1, [0, 1], None, 0.0) == -1
    assert f.prep_step(0, 0, [(0, 1)], 1, 2, 3, 0, 4, 8, 1.0, 0.0, 0, 0, 1e-6, 0.0, True, 0) == -1


@pytest.mark.parametrize("missing", ["g++", "Python.h"])
def test_a_build_without_what_the_front_module_needs(monkeypatch, tmp_path, capfd, missing):
    from __graft_entry__ import _load_builder

    build = _load_builder()
    built = tmp_path / "front.so"
    built.write_bytes(b"of an older source")
    monkeypatch.setattr(build, "FRONT_PATH", str(built))
    if missing == "g++":
        monkeypatch.setattr(build.shutil, "which", lambda name: None)
    else:
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build_front() is None
    assert f"{missing} not found" in capfd.readouterr().err and not built.exists()


def test_both_builds_of_the_library_bring_the_front_module(monkeypatch, tmp_path):
    from __graft_entry__ import _load_builder

    build, made = _load_builder(), []
    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path / "build"))
    monkeypatch.setattr(build, "sources", lambda: ["one.hip"])
    monkeypatch.setattr(build.subprocess, "run", lambda *a, **kw: type("Done", (), {"returncode": 0, "stderr": ""}))
    monkeypatch.setattr(build, "build_front", lambda: made.append(1))
    build.build(), build.build(timeline=True)
    assert made == [1, 1]


@gpu
def test_steps_without_the_front_module_give_the_same(monkeypatch):
    P, rng = pkg(), np.random.default_rng(3)
    front()
    q, k, v = normal(rng, 1, 8 * 128), normal(rng, 1, 256), normal(rng, 1, 256)
    d = [torch.from_numpy(x).cuda() for x in (q, k, v)]
    outs = []
    for f in (P.hip_compute._front, P._native.NoFront):
        monkeypatch.setattr(P.hip_compute, "_front", f)
        pool = P.KvPool(1, 2, 128, capacity_rows=64)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        cache, out = pool.acquire(), torch.full_like(d[0], float("nan"))
        for _ in range(3):
            pool.attention_step_device(0, [(cache, 1)], *(x.data_ptr() for x in d), out.data_ptr(), 8)
            pool.attention_prep_step_device(0, [(cache, 1)], *(x.data_ptr() for x in d), out.data_ptr(), 8, rope_base=1e4)
        pool.truncate([cache], [5])
        outs += [out.cpu().numpy(), P.gqa_attention(q, 1, 8, [4], cache.view(0))]
        pool.close()
    assert np.array_equal(outs[0], outs[2]) and np.array_equal(outs[1], outs[3])


@gpu
@pytest.mark.parametrize("slots", [1, 3, 65])
def test_both_ways_of_a_step_give_the_same(slots):
    P, rng = pkg(), np.random.default_rng(slots)
    outs = []
    rows, q_heads, kv_heads, d = [1 + i % 2 for i in range(slots)], 8, 2, 128
    n = sum(rows)
    k0, v0 = normal(rng, slots * 40, kv_heads * d), normal(rng, slots * 40, kv_heads * d)
    q, k, v, gate = (normal(rng, n, w * d) for w in (q_heads, kv_heads, kv_heads, q_heads))
    norm = 1 + 0.1 * normal(rng, d)
    t = {name: torch.from_numpy(np.ascontiguousarray(a)).cuda() for name, a in
         dict(k0=k0, v0=v0, q=q, k=k, v=v, gate=gate, norm=norm.reshape(-1)).items()}
    at = {name: x.data_ptr() for name, x in t.items()}
    for plain in (True, False):
        pool = P.KvPool(2, kv_heads, d, max_slots=slots, capacity_rows=64)
        pool.set_stream(torch.cuda.current_stream().cuda_stream)
        caches = [pool.acquire() for _ in range(slots)]
        for layer in range(2):
            pool.append_device(layer, [(c, 40) for c in caches], at["k0"], at["v0"])
        items = list(zip(caches, rows))
        lengths = [33] * slots
        if not plain:
            items, lengths = Indexed([(np.uint32(c.slot) if i % 2 else c, np.int64(r)) for i, (c, r) in enumerate(items)]), \
                np.array(lengths)
        pool.truncate(caches if plain else [np.uint32(c.slot) for c in caches], lengths)
        out = torch.full_like(t["q"], float("nan"))
        both = torch.full_like(t["q"], float("nan"))
        pool.attention_step_device(0, items, at["q"], at["k"], at["v"], out.data_ptr(), q_heads, softcap=30)
        pool.attention_prep_step_device(1, items, at["q"], at["k"], at["v"], both.data_ptr(), q_heads,
                                        q_norm_ptr=at["norm"], k_norm_ptr=at["norm"], rope_base=1e4, gate_ptr=at["gate"],
                                        interleaved=False if plain else 0, rotary_dim=64)
        torch.cuda.synchronize()
        outs.append((out.cpu().numpy(), both.cpu().numpy(), [c.stored_len(0) for c in caches]))
        with pytest.raises(P.AttentionError) as e:
            pool.attention_step_device(7, items, at["q"], at["k"], at["v"], out.data_ptr(), q_heads)
        assert e.value == P.AttentionError("InvalidLayer", layer=7, layer_count=2)
        pool.close()
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])
    assert np.isfinite(outs[0][0]).all() and np.isfinite(outs[0][1]).all()
    assert outs[0][2] == outs[1][2] == [33 + r for r in rows]


@gpu
def test_both_ways_of_the_host_calls_give_the_same():
    P, rng = pkg(), np.random.default_rng(5)
    q_heads, kv_heads, d, rows = 8, 2, 64, 5
    cfg = P.GlimmerConfig(layers=[P.LayerKind.Global], q_heads=q_heads, kv_heads=kv_heads, key_length=d, value_length=d)
    q, k, v = (normal(rng, rows, w * d) for w in (q_heads, kv_heads, kv_heads))
    outs = []
    for odd in (lambda x: x, lambda x: x.astype(np.float64), lambda x: np.repeat(x, 2, axis=0)[::2], lambda x: x.tolist()):
        compute = P.HipCompute(elem="f32", capacity_rows=64)
        outs.append(compute.attention(P.AttentionRequest(odd(q), odd(k), odd(v), 0, P.LayerKind.Global, cfg), P.PositionCache()))
        cache = compute.kv_cache()
        positions = list(range(rows))
        outs.append(P.gqa_attention(odd(q), rows, q_heads, positions, cache.view(0)))
        outs.append(P.gqa_attention(odd(q), rows, q_heads, np.array(positions), cache.view(0), P.AttentionParams(scale=d ** -0.5)))
        with pytest.raises(P.AttentionError):
            P.gqa_attention(odd(q), rows + 1, q_heads, positions, cache.view(0))
    assert all(x.dtype == np.float32 and x.shape == (rows * q_heads * d,) for x in outs)
    for x in outs[3:]:
        assert np.array_equal(x, outs[0]) or np.array_equal(x, outs[1]) or np.array_equal(x, outs[2])
    for i in range(3):
        assert all(np.array_equal(outs[i], x) for x in outs[i::3])
