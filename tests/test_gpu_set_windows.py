"""Sets whose radix tiles hold as many sketches as the tile's window of offsets, one more
and one less."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, zipf_keys

pytestmark = pytest.mark.gpu

TILE, WINDOW = 4096, 128


@pytest.mark.parametrize("per", [TILE // (WINDOW - 1), TILE // WINDOW, TILE // (WINDOW + 1), TILE // (WINDOW // 2), 1])
def test_tiles_of_many_sketches(gpu, per):
    import qsketch_amd as q
    print("CASE set window", per, flush=True)
    ns = 900
    lengths = np.full(ns, per)
    lengths[::7] = 0
    lengths[5] += 600
    offs = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    low = [1, 13, 61]
    S = q.SketchSet([q.make_params(low[i % 3], 8, n_masks=61, rng_seed=i + 1) for i in range(ns)])
    batches = [zipf_keys(2.0, 1 << 9, int(offs[-1]), s) for s in range(4)]
    for b in batches:
        S.insert(to_dev(b), offs)
    for i in range(ns):
        o = po.OracleSketch(low[i % 3], 8, 61, rng_seed=i + 1)
        for b in batches:
            part = b[int(offs[i]):int(offs[i + 1])]
            if part.size:
                assert o.insert(part) == 0
        st = S.export_state(i)
        assert np.array_equal(st["low"], o.low()) and np.array_equal(st["high"], o.high()), i
        assert st["next"] == o.next, i
