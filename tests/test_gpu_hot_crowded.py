"""A filtered insert whose sample crowds the candidate count: most of its keys hash to two
of the 256 bins, which hold far more distinct keys than the block's table has slots."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import to_dev, to_host_u32, uniform_keys

pytestmark = pytest.mark.gpu

N = (1 << 26) + 4097


def test_crowded_candidates_never_show_in_the_result(gpu):
    import qsketch_amd as q
    print("CASE hot crowded", flush=True)
    a = np.arange(1 << 24, dtype=np.uint64)
    two_bins = a[((a * 0x9E3779B1) & 0xFFFFFFFF) >> 24 < 2].astype(np.uint32)  # the sample's own hash
    rs = np.random.default_rng(11)
    keys = uniform_keys(N, 5)
    m = rs.random(N)
    frequent = m < 0.5
    keys[frequent] = rs.choice(two_bins[:6000], int(frequent.sum()))
    filling = (m >= 0.5) & (m < 0.75)
    keys[filling] = rs.choice(two_bins[6000:66000], int(filling.sum()))
    dk = to_dev(keys)
    uq = to_dev(np.unique(keys[: 1 << 22]))
    out = []
    for hot in (True, False):
        g = q.Sketch_GPU_Sub_Warp_Level(q.number_of_buckets(1 << 24), 8, 1 << 18, 32, rng_seed=1)
        g.set_hot_filter(hot)
        g.insert(dk)
        st = g.export_state()
        out.append((st["low"], st["high"], st["next"], to_host_u32(g.search(uq)), g.stats()["hot_keys"]))
        g.destroy()
    assert out[0][4] > 0 == out[1][4]  # the filter ran, and only where it was on
    for x, y in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(x, y)
