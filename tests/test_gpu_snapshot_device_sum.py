"""Version 1 snapshots whose checksum is the device's: capture and load at the payload sizes where
the split of the walk can go wrong (below and above the size from which the device sums, tails that
are no whole run, one workgroup's runs more or less, several pieces), against the host's byte walk."""
import struct

import numpy as np
import pytest

from helpers import normal, pkg

pytestmark = pytest.mark.gpu

# layers, kv heads, head dim, window, rows: payload = layers * rows * 2 * heads * dim * 4 bytes
SHAPES = [
    (1, 1, 5, 0, 3276),      # 131,040 bytes: the host's walk
    (1, 1, 5, 0, 3277),      # 131,080: 2,048 runs and 8 bytes
    (2, 1, 8, 0, 1032),      # 132,096: 8 workgroups of runs and 16 runs
    (3, 2, 16, 100, 900),    # rings that have wrapped
    (1, 1, 7, 0, 65537),     # 3.67 MB, 56 bytes to the row
    (2, 4, 128, 0, 4500),    # 36.9 MB: a second piece, ragged
]


@pytest.mark.parametrize("elem", ["f16", "f32"])
@pytest.mark.parametrize("layers,heads,dim,window,rows", SHAPES)
def test_capture_and_load_against_the_hosts_walk(layers, heads, dim, window, rows, elem):
    P = pkg()
    rng = np.random.default_rng(rows + dim)
    pattern = [P.LayerKind.windowed(window) if window and i % 2 == 0 else P.LayerKind.Global for i in range(layers)]
    pool = P.KvPool(pattern, heads, dim, elem=elem, max_slots=2, capacity_rows=rows + 4)
    cache = pool.acquire()
    for layer, kind in enumerate(pattern):
        first = max(0, rows - window) if kind.is_windowed else 0
        k, v = normal(rng, rows - first, heads * dim), normal(rng, rows - first, heads * dim)
        cache.restore_bulk(layer, first, k, v)
    data = P.capture_bytes(cache, "a model")
    assert struct.unpack("<Q", data[-8:])[0] == P.checksum(data[:-8])
    snapshot = P.KvSnapshot.from_bytes(data)
    for layer in range(layers):
        _, k, v = cache.view(layer).rows()
        if elem == "f16":
            k, v = k.view(np.float16).astype(np.float32), v.view(np.float16).astype(np.float32)
        assert np.array_equal(snapshot.layers[layer].keys, k.reshape(-1))
        assert np.array_equal(snapshot.layers[layer].values, v.reshape(-1))

    other = P.restore_bytes(pool, data, "a model")
    for layer in range(layers):
        for a, b in zip(other.read_rows(layer, 0, other.stored_len(layer)), cache.read_rows(layer, 0, cache.stored_len(layer))):
            assert np.array_equal(a, b)
    other.release_slot()
    for at in (len(data) - 9, len(data) // 2):  # the last payload byte, one in the middle
        bad = bytearray(data)
        bad[at] ^= 0x20
        with pytest.raises(P.KvError) as e:
            P.restore_bytes(pool, bytes(bad))
        assert e.value.variant == "ChecksumMismatch"
    pool.close()
