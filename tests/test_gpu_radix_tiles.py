"""Inserts at the edges of the radix passes: around one tile of 4096 items, around
the most tiles that a scatter sums by itself (64), and digits of one bit up to
8, in one to four passes, the last one narrower than the others or not."""
from __future__ import annotations

import pytest

from tests.helpers import assert_same_state, make_pair, to_dev, zipf_keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("n_low", [1, 2, 251, 257, 131071, 200003, 1 << 20, (1 << 24) + 43])
@pytest.mark.parametrize("n", [4097, 8191, 64 * 4096, 64 * 4096 + 1])
def test_radix_edges(gpu, n, n_low, key_bytes):
    print("CASE radix", n, n_low, key_bytes, flush=True)
    import numpy as np
    g, o = make_pair(n_low, n_high=1 << 12, key_bytes=key_bytes)
    keys = zipf_keys(0.9, 1 << 18, n, 3)
    if key_bytes == 8:
        keys = keys.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    g.insert(to_dev(keys))
    assert o.insert(keys) == 0
    assert_same_state(g, o, f"n={n} n_low={n_low}")
