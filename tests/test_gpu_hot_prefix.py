"""Filtered inserts at call lengths where the prefix is at its least, in between
and at its most: the same state as the ordered insert."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import to_host_u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1 << 26, (1 << 26) + 16 * 1024 + 5, (5 << 25) + 3, (1 << 28) + 31])
def test_filtered_equals_ordered_at_prefix_edges(gpu, n):
    import torch
    import qsketch_amd as q
    print("CASE prefix", n, flush=True)
    keys = q.Zipf(1.2, 1 << 20).keys_u32(seed=n & 0xffff, n=n)
    seen = torch.unique(keys[: 1 << 22])
    got = []
    for hot in (True, False):
        g = q.Sketch_GPU_Sub_Warp_Level(q.number_of_buckets(1 << 24), 8, 1 << 19, 32, rng_seed=1)
        g.set_hot_filter(hot)
        g.insert(keys)
        st = g.export_state()
        got.append((st["low"], st["high"], st["next"], to_host_u32(g.search(seen)), g.stats()["hot_keys"]))
        g.destroy()
    assert got[0][4] > n // 4 and got[1][4] == 0
    for a, b in zip(got[0][:4], got[1][:4]):
        assert np.array_equal(a, b)
