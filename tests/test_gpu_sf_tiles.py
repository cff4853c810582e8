"""Unsorted SF inserts at the edges of their tiles: 256 keys (one per thread), and 2048 for
long calls into a sketch of one bucket."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, to_host_u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["distinct", "zipf", "one"])
@pytest.mark.parametrize("key_bytes,n,n_buckets", [
    (4, 255, 3067), (4, 256, 3067), (4, 257, 3067), (8, 256 * 7 + 1, 3067), (4, 1 << 17, 1), (4, (1 << 17) + 1, 1),
    (8, (1 << 17) + 2047, 1),
])
def test_sf_unsorted_tiles(gpu, key_bytes, n, n_buckets, kind):
    import qsketch_amd as q
    print("CASE sf tiles", key_bytes, n, n_buckets, kind, flush=True)
    dt = np.uint32 if key_bytes == 4 else np.uint64
    if kind == "distinct":
        keys = (np.arange(n, dtype=np.uint64) * 2654435761 & 0xFFFFFFFF).astype(dt)
    elif kind == "zipf":
        keys = q.Zipf(1.2, 1 << 12, device=False).keys_u32_host(n, n).astype(dt)
    else:
        keys = np.full(n, 12345, dt)
    keys[::5] = np.iinfo(dt).max  # the tile table's empty marker
    g = q.Sketch_GPU_SF_Host_Sub_Warp(n_buckets, 8, 3, 1, 1021, key_bytes=key_bytes, rng_seed=11)
    o = po.OracleSF(n_buckets, 8, 3, 1021, key_bytes=key_bytes, rng_seed=11)
    for part in (keys, keys[: n // 2 + 1]):
        g.insert(to_dev(part))
        o.insert(part)
        st = g.export_state()
        assert np.array_equal(st["split"], o.split())
        assert np.array_equal(st["search"], o.search())
    uq = np.unique(keys)
    assert np.array_equal(to_host_u32(g.search(to_dev(uq))), o.query(uq))
