"""A stream-ordered batched lookup answers every key of the call, also those before
the first offset (the first sketch's) and after the last one (the last sketch's)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.helpers import to_dev, to_host_u32, zipf_keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("more", [0, 1 << 19])  # short batches, and those that are cut into tiles
@pytest.mark.parametrize("offs", [[0, 3000, 5000, 9000], [700, 3000, 3000, 8000], [1500, 1500, 1500, 1500],
                                  [9000, 9000, 9000, 9000]])
def test_every_key_is_answered(gpu, offs, more):
    import torch
    import qsketch_amd as q
    print("CASE query span", offs, more, flush=True)
    offs = [offs[0], offs[1], offs[2] + more // 2, offs[3] + more // 2]
    n, ns = 9000 + more, 3
    S = q.SketchSet([q.make_params(1021, 512, rng_seed=i + 1) for i in range(ns)])
    m = 9000
    keys = zipf_keys(1.1, 1 << 10, ns * m, 1)
    S.insert(to_dev(keys), np.arange(ns + 1, dtype=np.uint64) * np.uint64(m))
    ask = zipf_keys(1.1, 1 << 11, n, 2)
    d_offs = to_dev(np.array(offs, np.uint64))
    out = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    S.search_async(to_dev(ask), d_offs, n, out)
    torch.cuda.synchronize()
    got = to_host_u32(out)
    part = np.clip(np.searchsorted(offs, np.arange(n), side="right") - 1, 0, ns - 1)
    for i in range(ns):
        o = po.OracleSketch(1021, 512, 1021, rng_seed=i + 1)
        assert o.insert(keys[i * m:(i + 1) * m]) == 0
        assert np.array_equal(got[part == i], o.query(ask[part == i])), i
