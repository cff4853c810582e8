"""Batched inserts whose sketches begin and end on the edges of the first radix
pass's tiles (4096 keys, and halves of them): tiles of one sketch, of several, of more than the window of
64 holds, empty sketches between them, and sets that the search for a tile's
sketches takes one, two and three rounds of 64 offsets to search."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, zipf_keys

pytestmark = pytest.mark.gpu

LENGTHS = {
    "edges": [2048, 1, 2047, 4096, 0, 2049, 0, 0, 2047, 6143, 1],
    "edges_whole": [4096, 1, 4095, 8192, 0, 4097, 0, 0, 4095, 12287, 1],
    "window_63_64_65": [32] * 64 + [2048] + [31] * 64 + [64] + [31, 30] * 33 + [33],
    "window_whole": [64] * 64 + [4096] + [63] * 64 + [64] + [63, 62] * 33 + [65],
    "two_rounds": [0] * 63 + [5000] + [0] * 200 + [3000, 1, 0, 4095] + [7] * 300,
    "three_rounds": [1] * 2100 + [0] * 1500 + [4100, 0, 2] + [1] * 700,
}


@pytest.mark.parametrize("chunk_keys", [0, 3001])
@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("kind", sorted(LENGTHS))
def test_batched_insert_tiles(gpu, kind, key_bytes, chunk_keys):
    import qsketch_amd as q
    print("CASE multi tiles", kind, key_bytes, chunk_keys, flush=True)
    lengths = LENGTHS[kind]
    lows, masks = [13, 61, 1021, 4093], [1021, 509, 61]
    S = q.SketchSet([q.make_params(lows[i % 4], 64, n_masks=masks[i % 3], key_bytes=key_bytes, rng_seed=i + 1,
                                   chunk_keys=chunk_keys if i == 0 else 0) for i in range(len(lengths))])
    parts = [zipf_keys(1.1, 1 << 10, n, 7 + i) if n else np.zeros(0, np.uint32) for i, n in enumerate(lengths)]
    if key_bytes == 8:
        parts = [p.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15) for p in parts]
    offs = np.zeros(len(parts) + 1, np.uint64)
    offs[1:] = np.cumsum([p.size for p in parts])
    S.insert(to_dev(np.concatenate(parts)), offs)
    for i, p in enumerate(parts):
        if p.size == 0:
            continue
        if i > 400 and i % 97 and p.size < 2048:
            continue
        o = po.OracleSketch(lows[i % 4], 64, masks[i % 3], key_bytes=key_bytes, rng_seed=i + 1)
        assert o.insert(p) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()) and np.array_equal(st["high"], o.high()), i
        assert st["next"] == o.next, i
