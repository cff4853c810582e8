"""Sets on both sides of the number of sketches from which the closing kernel moves the
allocators on by the allocations instead of sketch by sketch."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, zipf_keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1024, 1025, 3001])
@pytest.mark.parametrize("chunk_keys", [0, 50000])
def test_allocators_of_large_sets(gpu, ns, chunk_keys):
    import qsketch_amd as q
    print("CASE large set", ns, chunk_keys, flush=True)
    rs = np.random.default_rng(ns)
    lengths = rs.integers(0, 400, ns)
    lengths[rs.integers(0, ns, 20)] = 3000  # many allocations in one sketch
    lengths[-1] = 700
    offs = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    low = [1, 3, 13, 61]
    S = q.SketchSet([q.make_params(low[i % 4], 64, n_masks=61, rng_seed=i + 1, chunk_keys=chunk_keys if i == 0 else 0)
                     for i in range(ns)])
    batches = [zipf_keys(a, 1 << 9, int(offs[-1]), s) for a, s in ((1.3, 1), (1.1, 2))]
    for b in batches:
        S.insert(to_dev(b), offs)
    linked = 0
    for i in range(ns):
        o = po.OracleSketch(low[i % 4], 64, 61, rng_seed=i + 1)
        for b in batches:
            part = b[int(offs[i]):int(offs[i + 1])]
            if part.size:
                assert o.insert(part) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()) and np.array_equal(st["high"], o.high()), i
        assert st["next"] == o.next, i
        linked += o.next - 1025
    assert S.stats()["linked_buckets"] == linked > ns // 6


def test_full_pool_in_a_large_set(gpu):
    import qsketch_amd as q
    print("CASE large set, full pool", flush=True)
    ns, per = 1500, 1500
    S = q.SketchSet([q.make_params(13, 2, n_masks=61, rng_seed=i + 1) for i in range(ns)])
    offs = np.arange(ns + 1, dtype=np.uint64) * np.uint64(per)
    with pytest.raises(q.QSketchError) as e:
        S.insert(to_dev(zipf_keys(1.5, 1 << 8, ns * per, 1)), offs)
    assert e.value.code == q.QS_ERR_POOL
    S.clear()
    keys = zipf_keys(1.1, 1 << 8, ns * 20, 2)
    S.insert(to_dev(keys), np.arange(ns + 1, dtype=np.uint64) * np.uint64(20))
    for i in range(0, ns, 97):
        o = po.OracleSketch(13, 2, 61, rng_seed=i + 1)
        assert o.insert(keys[i * 20:(i + 1) * 20]) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()) and st["next"] == o.next, i
