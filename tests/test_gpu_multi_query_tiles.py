"""Batched lookups at the length from which they are cut into tiles, with parts on the
edges of that split: tiles of 1024 keys, tiles of 8 or more sketches, parts of 256
keys, empty parts."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, to_host_u32, zipf_keys

pytestmark = pytest.mark.gpu

TILES_MIN = 1 << 19
READS = {
    "ragged": [1, 0, 255, 256, 257, 1023, 0, 0, 1024, 1025, 3000, 5],
    "tiny": [3, 0, 1, 7] * 80 + [2000] + [1] * 9,
    "seven_and_eight": [146] * 7 + [2] + [128] * 8 + [5000] + [127] * 9,
    "one": [0, 0, 70001, 0],
}


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("n", [TILES_MIN - 1, TILES_MIN, TILES_MIN + 1025])
@pytest.mark.parametrize("kind", sorted(READS))
def test_long_batched_lookup_parts(gpu, kind, n, key_bytes):
    import qsketch_amd as q
    print("CASE multi query tiles", kind, n, key_bytes, flush=True)
    reads = list(READS[kind])
    reads.insert(len(reads) // 2, n - sum(reads))  # the rest of the batch, between the small parts
    ns = len(reads)
    lows, masks = [13, 61, 1021, 4093], [1021, 509, 61]
    S = q.SketchSet([q.make_params(lows[i % 4], 2048, n_masks=masks[i % 3], key_bytes=key_bytes, rng_seed=i + 1)
                     for i in range(ns)])
    lengths = np.random.default_rng(ns).integers(0, 900, ns)
    lengths[ns // 2] = 20000

    def keys(m, seed):
        k = zipf_keys(1.1, 1 << 10, int(m), seed) if m else np.zeros(0, np.uint32)
        return k.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15) if key_bytes == 8 else k

    ins = [keys(m, 1000 + i) for i, m in enumerate(lengths)]
    ask = [keys(m, 5000 + i) for i, m in enumerate(reads)]
    offs = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    qoffs = np.concatenate([[0], np.cumsum(reads)]).astype(np.uint64)
    S.insert(to_dev(np.concatenate(ins)), offs)
    est = to_host_u32(S.search(to_dev(np.concatenate(ask)), qoffs))
    for i in range(ns):
        o = po.OracleSketch(lows[i % 4], 2048, masks[i % 3], key_bytes=key_bytes, rng_seed=i + 1)
        if ins[i].size:
            assert o.insert(ins[i]) == 0
        if reads[i]:
            assert np.array_equal(est[int(qoffs[i]):int(qoffs[i + 1])], o.query(ask[i])), i
