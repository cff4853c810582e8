"""Chunks at the edges of the radix scan: 64 tiles of 4096 keys (no scan), 16 groups of 16
tiles (the scatter sums the groups itself), one tile more."""
from __future__ import annotations

import pytest

from tests.helpers import assert_same_state, make_pair, to_dev, zipf_keys

pytestmark = pytest.mark.gpu

TILE = 4096


@pytest.mark.parametrize("n", [64 * TILE, 64 * TILE + 1, 240 * TILE + 1, 256 * TILE, 256 * TILE + 1])
def test_scan_of_the_tile_counts(gpu, n):
    print("CASE radix groups", n, flush=True)
    keys = zipf_keys(1.1, 1 << 16, n, seed=n)
    g, o = make_pair(100003, n_high=1 << 12)
    for part in (keys, keys[::-1].copy()):
        g.insert(to_dev(part))
        assert o.insert(part) == 0
        assert_same_state(g, o, f"n={n}")
