"""Filtered inserts whose samples are unlike a Zipf stream: which keys the filter
picks must never show in the result."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import make_pair, to_dev, to_host_u32, uniform_keys

pytestmark = pytest.mark.gpu

N = (1 << 26) + 4097
SAMPLE = 1 << 20


def _keys(kind):
    rs = np.random.default_rng(11)
    keys = uniform_keys(N, 5)
    if kind == "one":          # a single key fills the sample and most of the stream
        keys[rs.random(N) < 0.9] = np.uint32(12345)
        keys[:SAMPLE] = np.uint32(12345)
    elif kind == "empty":      # the table's empty marker is the hottest key
        keys[rs.random(N) < 0.5] = np.uint32(0xFFFFFFFF)
        keys[::3] = rs.integers(0, 500, keys[::3].size).astype(np.uint32)
    elif kind == "ties":       # more candidates than the table takes, all equally frequent
        keys[:] = (rs.integers(0, 20000, N) * 2654435761 & 0xFFFFFFFF).astype(np.uint32)
        keys[:SAMPLE] = (np.arange(SAMPLE) % 20000 * 2654435761 & 0xFFFFFFFF).astype(np.uint32)
    elif kind == "crowded":    # the frequent keys of the sample share few bins of its hash
        hot = np.arange(1 << 22, dtype=np.uint64) * 2654435769 & 0xFFFFFFFF
        hot = np.nonzero(hot >> 24 < 2)[0].astype(np.uint32)
        keys[::2] = rs.choice(hot[:30000], keys[::2].size)
    return keys


@pytest.mark.parametrize("kind", ["one", "empty", "ties", "crowded"])
def test_filtered_insert_equals_ordered_insert(gpu, kind):
    import qsketch_amd as q
    print("CASE hot", kind, flush=True)
    keys = _keys(kind)
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
    assert out[1][4] == 0
    if kind != "crowded":
        assert out[0][4] > 0  # the filter ran
    for a, b in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(a, b)
