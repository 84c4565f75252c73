"""Version 2 snapshots, whose trailer joins the sums of the file's 1 MiB blocks: capture and load with the blocks' sums
made on the device, against the host's walk. Payloads below and above the size from which the device sums; headers of any
length, so that blocks begin and end anywhere in a run of 64 bytes and rows; one block, the next begun by a few
bytes, several pieces."""
import struct

import numpy as np
import pytest

from helpers import normal, pkg

pytestmark = pytest.mark.gpu

MB = 1 << 20
# layers, kv heads, head dim, window, rows: payload = layers * rows * 2 * heads * dim * 2 bytes
SHAPES = [
    (1, 1, 5, 0, 6550),      # 131,000 bytes: the host's walk
    (1, 1, 5, 0, 6554),      # 131,080
    (2, 1, 8, 0, 16380),     # a block less 320 bytes: the header's length says whether a second begins
    (1, 1, 7, 0, 37444),     # a block less 144
    (3, 2, 16, 700, 9000),   # rings that have wrapped; three blocks
    (2, 4, 128, 0, 8500),    # 34.8 MB: a second piece, ragged
]


@pytest.mark.parametrize("name", ["", "m", "a model of another name" * 3])
@pytest.mark.parametrize("layers,heads,dim,window,rows", SHAPES)
def test_capture_and_load_against_the_hosts_walk(layers, heads, dim, window, rows, name):
    P = pkg()
    rng = np.random.default_rng(rows + dim)
    pattern = [P.LayerKind.windowed(window) if window and i % 2 == 0 else P.LayerKind.Global for i in range(layers)]
    pool = P.KvPool(pattern, heads, dim, elem="f16", max_slots=2, capacity_rows=rows + 4)
    cache = pool.acquire()
    for layer, kind in enumerate(pattern):
        first = max(0, rows - window) if kind.is_windowed else 0
        k, v = normal(rng, rows - first, heads * dim), normal(rng, rows - first, heads * dim)
        cache.restore_bulk(layer, first, k, v)
    data = P.capture_bytes(cache, name, elem="f16")
    assert struct.unpack("<Q", data[-8:])[0] == P.checksum_blocks(data[:-8])
    other = P.restore_bytes(pool, data, name)
    for layer in range(layers):
        for a, b in zip(other.read_rows(layer, 0, other.stored_len(layer)), cache.read_rows(layer, 0, cache.stored_len(layer))):
            assert np.array_equal(a, b)
    other.release_slot()
    payload = layers * 2 * heads * dim * 2 * rows if not window else 0
    first = len(data) - 8 - payload
    for at in (len(data) - 9, len(data) // 2, *((first, MB - 1, MB) if payload > MB else ())):
        if at >= len(data) - 8:
            continue
        bad = bytearray(data)
        bad[at] ^= 0x20
        with pytest.raises(P.KvError) as e:
            P.restore_bytes(pool, bytes(bad))
        assert e.value.variant == "ChecksumMismatch"
    pool.close()
