"""A failed allocation is reported once, by the call that made it: what follows on the
device is not told of it again."""
from __future__ import annotations

import pytest

from tests.helpers import assert_same_state, make_pair, to_dev, uniform_keys

pytestmark = pytest.mark.gpu


def test_calls_after_a_failed_allocation_work(gpu):
    import torch
    import qsketch_amd as q
    print("CASE alloc failure", flush=True)
    g, o = make_pair(1021)
    keys = uniform_keys(5000, 3)
    dk = to_dev(keys)
    with pytest.raises(q.QSketchError) as e:  # two tables of 256 GiB each
        q.Sketch_GPU_SF_Host_Sub_Warp(4294967291, 16, 1)
    assert e.value.code == q.QS_ERR_NOMEM
    g.insert(dk)
    assert o.insert(keys) == 0
    assert_same_state(g, o)
    assert int(torch.arange(5, device="cuda").sum()) == 10
