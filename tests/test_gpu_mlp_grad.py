"""Gradients of the learned form's network at batch sizes on the edges of the
kernel's work split (groups of 16 keys, 256 blocks), against the float64 oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import mlp_oracle as mo
from tests.helpers import to_dev
from tests.test_gpu_learned import _exact_params, _grad_abs_sums, _keys, _learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4096, 4097, 9001])
def test_gradient_elements_within_their_rounding(gpu, n):
    """On the exact network the forward is exact, so each element must equal
    the oracle within the rounding of its own FP32 sum: (2n + 256) u times
    the sum of the magnitudes of its terms, whatever the order."""
    import torch
    print("CASE grad", n, flush=True)
    L = _learned()
    p = _exact_params(12)
    L.set_params(p)
    keys = _keys(n, 100 + n)
    t = (np.random.default_rng(n).integers(-96, 97, n) / 32).astype(np.float32)
    loss, g = L.grad(to_dev(keys), torch.from_numpy(t).cuda())
    rl, rg = mo.grad(p, keys, t, exact=True)
    u = 2.0 ** -24
    bound = (2 * n + 256) * u * _grad_abs_sums(p, keys, t.astype(np.float64))
    assert np.all(np.abs(g.astype(np.float64) - rg) <= bound)
    y, _ = mo.forward(p, keys, exact=True)
    assert abs(loss - rl) <= (n + 8) * u * 0.5 * np.mean((y - t) ** 2) + 1e-30
    # a step applies the same gradient: Adam's first step from zero moments
    # moves every element with a gradient well above eps by lr
    L.step(to_dev(keys), torch.from_numpy(t).cuda(), lr=2.0 ** -7, eps=0.0, want_loss=False)
    moved = L.get_params().astype(np.float64) - p.astype(np.float64)
    big = np.abs(rg) > 2 * bound + 1e-6
    assert big.any()
    assert np.allclose(moved[big], -np.sign(rg[big]) * 2.0 ** -7, rtol=0, atol=2.0 ** -7 * 64 * u + 2 * u)
