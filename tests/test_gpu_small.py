"""Short inserts (one block, one launch) at the edges of its work split and of
the length up to which they run that way, against the oracle's whole state."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import assert_same_state, make_pair, to_dev, to_host_u32, uniform_keys, zipf_keys

pytestmark = pytest.mark.gpu


def _keys(kind, n, seed):
    if kind == "one":
        return np.full(n, 77, np.uint32)
    if kind == "uniform":
        return uniform_keys(n, seed)
    return zipf_keys(1.2, 64, n, seed)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 130, 1023, 1024, 1025, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("kind,n_low", [("zipf", 61), ("one", 1021), ("uniform", 1 << 25), ("zipf", 1)])
def test_short_inserts_equal_the_oracle(gpu, n, kind, n_low):
    print("CASE small", n, kind, n_low, flush=True)
    for key_bytes, semantics in ((4, 0), (8, 1)):
        if n_low > 1 << 20 and key_bytes == 8:
            continue  # (one large table is enough)
        g, o = make_pair(n_low, n_high=256, key_bytes=key_bytes, semantics=semantics, rng_seed=5)
        total = None
        for call in range(4):
            k = _keys(kind, n, seed=call)
            if key_bytes == 8:
                k = k.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
            if call == 1:
                g.insert_noalloc(to_dev(k))
                g.sync()
            elif call == 2:
                g.insert_async(to_dev(k))
                g.sync()
            else:
                g.insert(to_dev(k))
            assert o.insert(k) == 0
            total = k if total is None else np.concatenate([total, k])
        assert_same_state(g, o, f"n={n} {kind}")
        assert g.stats()["keys_inserted"] == 4 * n
        uq = np.unique(total)
        assert np.array_equal(to_host_u32(g.search(to_dev(uq))), o.query(uq))
        g.clear()
        st = g.export_state()
        assert not st["low"].any() and not st["high"].any() and st["next"] == 1025


def test_short_insert_reports_a_full_pool(gpu):
    import qsketch_amd as q
    print("CASE small pool", flush=True)
    g = q.Sketch_GPU_Sub_Warp_Level(4093, 8, 3, 32, rng_seed=1)
    keys = np.repeat(np.arange(20, dtype=np.uint32) * 7919, 200)
    with pytest.raises(q.QSketchError) as e:
        g.insert(to_dev(keys))
    assert e.value.code == q.QS_ERR_POOL
    g.clear()
    g.insert(to_dev(keys[:200]))
    o = po.OracleSketch(4093, 3, 1021, rng_seed=1)
    assert o.insert(keys[:200]) == 0
    assert_same_state(g, o, "after clear")


def test_short_captured_insert_replays(gpu):
    import torch
    print("CASE small graph", flush=True)
    g, o = make_pair(509, n_high=512, rng_seed=2)
    buf = torch.zeros(1500, dtype=torch.int32, device="cuda")
    graph = g.capture_insert(buf)
    for i in range(5):
        k = zipf_keys(1.1, 128, 1500, seed=i)
        buf.copy_(to_dev(k))
        graph.launch()
        torch.cuda.synchronize()
        assert o.insert(k) == 0
        assert_same_state(g, o, f"replay {i}")


@pytest.mark.parametrize("lows", [[13], [1021, 7, 65521], [(1 << 21) + 11, 3]])
def test_clear_empties_every_table(gpu, lows):
    """Tables below and above the size that the runtime's fill clears."""
    import qsketch_amd as q
    print("CASE clear", lows, flush=True)
    S = q.SketchSet([q.make_params(m, 700, rng_seed=i + 1) for i, m in enumerate(lows)])
    keys = [zipf_keys(1.3, 512, 30000, seed=i) for i in range(len(lows))]
    offs = np.arange(len(lows) + 1, dtype=np.uint64) * np.uint64(30000)
    for _ in range(2):
        S.insert(to_dev(np.concatenate(keys)), offs)
        S.clear()
        for i in range(len(lows)):
            st = S.export_state(i)
            assert not st["low"].any() and not st["high"].any() and st["next"] == 1025
    S.insert(to_dev(np.concatenate(keys)), offs)
    for i, m in enumerate(lows):
        o = po.OracleSketch(m, 700, 1021, rng_seed=i + 1)
        assert o.insert(keys[i]) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()) and np.array_equal(st["high"], o.high()) and st["next"] == o.next
