"""A captured insert keeps its scratch: batches that would need a larger one are
refused while it lives, and its replays stay right afterwards."""
from __future__ import annotations

import pytest

from tests.helpers import assert_same_state, make_pair, to_dev, zipf_keys

pytestmark = pytest.mark.gpu


def test_larger_batches_refused_while_a_graph_lives(gpu):
    import torch
    import qsketch_amd as q
    print("CASE graph scratch", flush=True)
    g, o = make_pair(509, n_high=512, rng_seed=2)
    buf = torch.zeros(1500, dtype=torch.int32, device="cuda")
    graph = g.capture_insert(buf)
    large = torch.zeros(1 << 26, dtype=torch.int32, device="cuda")  # long enough for the hot-key filter
    for refused in (lambda: g.capture_insert(large[:5000]), lambda: g.insert(large[:5000]), lambda: g.insert(large)):
        with pytest.raises(q.QSketchError) as e:
            refused()
        assert e.value.code == q.QS_ERR_STATE
    for i in range(3):
        k = zipf_keys(1.1, 128, 1500, seed=i)
        buf.copy_(to_dev(k))
        graph.launch()
        torch.cuda.synchronize()
        assert o.insert(k) == 0
        assert_same_state(g, o, f"replay {i}")
