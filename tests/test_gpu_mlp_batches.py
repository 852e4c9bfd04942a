"""Batch sizes at the edges of the gradient's split reduction (64 samples per block, sixteen runs of blocks, four
chains) and of the pinned buffer that host batches pass through (65,536 rows)."""
import numpy as np
import pytest

import oracle_lib as ol
from frehg_amd import gpu
from gpu_common import say
from test_gpu_mlp import GROUPS, random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 64 * 16 + 1, 64 * 67, 65537])
def test_gradient_and_predictions_at_batch_edges(n):
    say(f"MLP batch n={n}")
    params, norm, x, y = random_case(40 + n % 97, n=n)
    ctx = gpu.Context(0)
    ctx.mlp_set_params(params, norm)
    for _ in range(2):  # the second call reuses the buffers
        loss, g = ctx.mlp_loss_grad(x, y)
        p = ctx.mlp_predict(x).astype(np.float64)
    lref, gref = ol.mlp_loss_grad(params, norm, x, y, bf16=True)
    ref = ol.mlp_predict(params, norm, x, bf16=True)
    # the tolerances of test_gpu_mlp.py, which allow for the BF16 roundings of the same operands; the
    # single sample's are not averaged: one BF16 rounding (2^-8) per layer and pass
    assert loss == pytest.approx(lref, rel=1e-3 if n > 1 else 2.0 ** -8)
    for name, (lo, hi) in GROUPS.items():
        scale = np.abs(gref[lo:hi]).max()
        assert np.abs(g[lo:hi] - gref[lo:hi]).max() <= (5e-3 if n > 1 else 6 * 2.0 ** -8) * scale, name
    assert np.abs(p - ref).max() <= 2e-3 * np.abs(ref).max()
