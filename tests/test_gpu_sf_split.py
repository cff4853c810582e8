"""SF inserts at the edges of their work split: tiles of 512 and 2048 unsorted keys
(with the all-ones key, which is the tile table's empty marker), and sorted calls
whose ranges are 64 keys long, longer, and more than the wavefronts."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, to_host_u32

pytestmark = pytest.mark.gpu

SORTED = 1 << 16


@pytest.mark.parametrize("key_bytes,times,n", [
    (4, 3, 1), (4, 3, 511), (4, 3, 512), (4, 2, 513), (8, 3, 512 * 9 + 1), (4, 4, SORTED - 1), (8, 5, SORTED - 1),
    (4, 3, SORTED), (8, 3, SORTED + 63), (4, 3, 4096 * 64), (4, 1, 4096 * 64 + 1), (4, 3, 4096 * 128 + 65),
    (4, 9, 8192 * 64 + 4097),
])
@pytest.mark.parametrize("n_buckets", [1, 3067, 98297])
def test_sf_work_split(gpu, key_bytes, times, n, n_buckets):
    import qsketch_amd as q
    print("CASE sf split", key_bytes, times, n, n_buckets, flush=True)
    rs = np.random.default_rng(n + times)
    dt = np.uint32 if key_bytes == 4 else np.uint64
    keys = q.Zipf(1.2, 1 << 15, device=False).keys_u32_host(n, n).astype(dt)
    keys[rs.integers(0, n, n // 8)] = rs.integers(0, 1 << 32, n // 8, dtype=np.uint64).astype(dt)  # rare ones
    keys[rs.integers(0, n, 1 + n // 50)] = np.iinfo(dt).max
    g = q.Sketch_GPU_SF_Host_Sub_Warp(n_buckets, 8, times, 1, 1021, key_bytes=key_bytes, rng_seed=11)
    o = po.OracleSF(n_buckets, 8, times, 1021, key_bytes=key_bytes, rng_seed=11)
    for part in (keys, keys[: n // 2 + 1]):
        g.insert(to_dev(part))
        o.insert(part)
        st = g.export_state()
        assert np.array_equal(st["split"], o.split())
        assert np.array_equal(st["search"], o.search())
    uq = np.unique(keys)
    assert np.array_equal(to_host_u32(g.search(to_dev(uq))), o.query(uq))


@pytest.mark.parametrize("n", [4096 * 65 - 1, 4096 * 65, 4096 * 449 - 63, 8192 * 512 + 4097])
def test_sf_most_ranges(gpu, n):
    """The most ranges of 64 keys, and the longest ranges, more than the wavefronts."""
    import qsketch_amd as q
    print("CASE sf ranges", n, flush=True)
    keys = q.Zipf(0.8, 1 << 20, device=False).keys_u32_host(n, n)
    g = q.Sketch_GPU_SF_Host_Sub_Warp(98297, 8, 3, 1, 1021, rng_seed=11)
    o = po.OracleSF(98297, 8, 3, 1021, rng_seed=11)
    g.insert(to_dev(keys))
    o.insert(keys)
    st = g.export_state()
    assert np.array_equal(st["split"], o.split())
    assert np.array_equal(st["search"], o.search())
