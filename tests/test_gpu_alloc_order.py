"""GPU parity of the allocation order: the ids of buckets promoted at chosen
stream positions, on the edges of the spans in which the insert counts them."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import assert_same_state, make_pair, to_dev, to_host_u32, uniform_keys

pytestmark = pytest.mark.gpu

SPAN = 8192  # chunk positions counted together


def _stream(n, at, seed):
    """n keys; the 130th insert of a key of its own falls on every position in
    `at` (the insert that finds its counters above 128), the other 129 on
    earlier ones; filler keys occur about once."""
    rs = np.random.default_rng(seed)
    keys = uniform_keys(n, seed)
    free = set(range(n)) - set(at)
    for i, p in enumerate(sorted(at)):
        before = np.array(sorted(x for x in free if x < p))
        take = rs.choice(before, 129, replace=False)
        free -= set(take.tolist())
        keys[take] = keys[p] = np.uint32(0xC0000000 + 7919 * i + seed)
    return keys


def _edges(n):
    near = [600, SPAN - 1, SPAN, SPAN + 1, SPAN + 31, SPAN + 32, 2 * SPAN - 1, 2 * SPAN, n - 2, n - 1]
    return sorted({p for p in near if 600 <= p < n})


@pytest.mark.parametrize("n", [2049, SPAN - 1, SPAN, SPAN + 1, 2 * SPAN + 1, 3 * SPAN - 2047])
@pytest.mark.parametrize("chunk_keys", [0, SPAN, 5000])
def test_ids_at_span_edges(gpu, n, chunk_keys):
    print("CASE", n, chunk_keys, flush=True)
    keys = _stream(n, _edges(n), seed=n)
    g, o = make_pair(12281, n_high=512, rng_seed=3, chunk_keys=chunk_keys)
    for part in (keys, keys[::-1].copy()):  # the second call finds linked buckets
        g.insert(to_dev(part))
        assert o.insert(part) == 0
        assert_same_state(g, o, f"n={n} chunk={chunk_keys}")
    assert o.next >= 1025 + len(_edges(n))
    uq = np.unique(keys)
    assert np.array_equal(to_host_u32(g.search(to_dev(uq))), o.query(uq))


@pytest.mark.parametrize("chunk_keys", [0, SPAN, 6001])
def test_set_ids_at_span_edges(gpu, chunk_keys):
    import qsketch_amd as q
    print("CASE set", chunk_keys, flush=True)
    lengths = [SPAN - 1, 0, 1, SPAN + 1, 3000, 2 * SPAN, 777]
    streams = [_stream(m, _edges(m), seed=50 + i) if m >= 700 else uniform_keys(m, 90 + i)
               for i, m in enumerate(lengths)]
    offs = np.zeros(len(lengths) + 1, np.uint64)
    offs[1:] = np.cumsum(lengths)
    S = q.SketchSet([q.make_params(4093, 256, rng_seed=i + 1, chunk_keys=chunk_keys if i == 0 else 0)
                     for i in range(len(lengths))])
    S.insert(to_dev(np.concatenate(streams)), offs)
    for i, k in enumerate(streams):
        o = po.OracleSketch(4093, 256, 1021, rng_seed=i + 1)
        if k.size:
            assert o.insert(k) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()), i
        assert np.array_equal(st["high"], o.high()), i
        assert st["next"] == o.next, i


# (also: 64 and 65 radix tiles, 16 and 17 groups of them, 64 and 65 spans)
@pytest.mark.parametrize("n", [64 * 2048, 64 * 2048 + 1, 64 * SPAN, 64 * SPAN + 1, 16 * 32 * 2048 + 1, 65537, (1 << 20) + 1, (1 << 21) - 255, (3 << 20) + 63])
def test_tail_windows_by_chunk_length(gpu, n):
    """Long runs cross the tail pass's windows, whose length follows the chunk's
    (256 items up to 2^20 keys, then more)."""
    from tests.helpers import zipf_keys
    print("CASE tail", n, flush=True)
    keys = zipf_keys(1.3, 1 << 14, n, seed=n)
    g, o = make_pair(12281, n_high=1 << 12)
    for part in (keys, keys[: n // 3]):
        g.insert(to_dev(part))
        assert o.insert(part) == 0
        assert_same_state(g, o, f"n={n}")
