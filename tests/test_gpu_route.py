"""Routing of the learned form at call lengths on the edges of its work split
(64-key steps, 1024-key chunks, 8-chunk groups, the length from which heavy
keys are grouped before they are counted), against exact counts and the sketch
oracle fed the light keys."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, to_host_u32

pytestmark = pytest.mark.gpu

GROUPED = 1 << 21


def _stream(n, key_bytes, seed):
    import qsketch_amd as q
    z = q.Zipf(1.1, 1 << 16, device=False)
    if key_bytes == 8:
        return z.keys_u64_noisy_host(seed, n, sigma=1.5)
    return z.keys_u32_host(seed, n)


@pytest.mark.parametrize("key_bytes,table_log2,n", [
    (8, 17, 1), (8, 17, 63), (8, 17, 64), (8, 17, 65), (8, 17, 1023), (8, 17, 1024), (8, 17, 1025),
    (8, 17, 8 * 1024 + 1), (4, 17, 5000), (8, 10, 70001), (8, 17, GROUPED - 1), (8, 17, GROUPED),
    (8, 17, GROUPED + 77), (4, 17, GROUPED + 1024), (8, 10, GROUPED + 5),
])
def test_route_at_work_split_edges(gpu, key_bytes, table_log2, n):
    import qsketch_amd as q
    print("CASE route", key_bytes, table_log2, n, flush=True)
    keys = _stream(n, key_bytes, 7 + n)
    if n > 100:
        keys[n // 2] = np.iinfo(keys.dtype).max  # (8 bytes: the empty-slot marker, never in the table)
    L = q.LearnedSketch(q.make_params(65537, 1 << 15, key_bytes=key_bytes, rng_seed=3), table_log2=table_log2)
    score = L.score(to_dev(keys)).cpu().numpy()
    L.threshold = float(np.quantile(score, 0.4))
    heavy = (score >= np.float32(L.threshold)) & ~((key_bytes == 8) & (keys == np.iinfo(np.uint64).max))
    o = po.OracleSketch(65537, 1 << 15, 1021, key_bytes=key_bytes, rng_seed=3)
    want = {}
    for part in (keys, keys[: max(1, n // 3)]):  # the second call finds the table filled
        h = heavy[: part.size]
        nh = L.insert(to_dev(part))
        tk, tc = L.table()
        held = h & np.isin(part.astype(np.uint64), tk)
        assert nh == int(held.sum())
        assert L.table_full or np.array_equal(held, h)
        for k, c in zip(*np.unique(part[held], return_counts=True)):
            want[int(k)] = want.get(int(k), 0) + int(c)
        if (~held).any():
            assert o.insert(part[~held]) == 0
        st = L.export_sketch_state()
        assert np.array_equal(st["low"], o.low()) and np.array_equal(st["high"], o.high())
        assert st["next"] == o.next
    assert dict(zip(tk.tolist(), tc.tolist())) == want
    uk = np.unique(keys)
    est = to_host_u32(L.search(to_dev(uk)))
    ref = o.query(uk)
    tab = np.isin(uk.astype(np.uint64), tk)
    assert np.array_equal(est[~tab], ref[~tab])
    assert all(want[int(k)] == int(e) for k, e in zip(uk[tab], est[tab]))
