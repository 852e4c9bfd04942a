"""Box shapes at the edges of the ensemble's tiles (256 columns along the rows, a row padded to a multiple
of 8 lanes): every box against the single-box GPU path with the same solver."""
import numpy as np
import pytest

from frehg_amd import abi, gpu, workloads
from gpu_common import say
from test_gpu_ensemble import single_box_heads

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 5), (1, 40, 17), (7, 3, 4), (8, 32, 3), (8, 33, 2), (9, 16, 9), (64, 4, 8), (65, 5, 9), (255, 2, 3),
          (256, 1, 6), (257, 1, 6)]


@pytest.mark.parametrize("precision,guess", [(abi.PREC_FP64, abi.GUESS_ZERO), (abi.PREC_FP64, abi.GUESS_EXTRAPOLATED),
                                             (abi.PREC_MIXED, abi.GUESS_EXTRAPOLATED)])
def test_boxes_at_the_edges_of_the_tiles(precision, guess):
    steps = 3
    case = workloads.EnsembleCase(nbox=len(SHAPES), seed=5, nxy=(2, 3), nz=(2, 3), precision=precision, guess=guess,
                                  rtol=1e-12)
    rng = np.random.default_rng(11)
    case.dims = list(SHAPES)
    case.ks = [1e-5 * np.exp(rng.standard_normal(nx * ny * nz)) for nx, ny, nz in SHAPES]
    ctx = gpu.Context(0)
    case.setup_gpu(ctx)
    for _ in range(steps):
        st = ctx.ens_step(use_graph=True)
        assert st.converged and st.max_rel_mass_residual <= 1e-10, st.max_rel_mass_residual
    # the tolerance of the comparison in test_gpu_ensemble.py: both solve each step to a relative residual
    # of 1e-12 (FP64; the mixed refinement's FP32 inner solves stop at other iterates), and only the
    # grouping of the sums differs
    tol = 1e-9 if precision == abi.PREC_FP64 else 1e-7
    for b, dims in enumerate(SHAPES):
        hs, ws = single_box_heads(case, b, steps, precision)
        hg, wg = ctx.ens_get(b, "h"), ctx.ens_get(b, "wc")
        say(f"box {dims}: |h - single-box GPU| {np.abs(hg - hs).max():.2e}")
        assert np.abs(hg - hs).max() <= tol * max(1.0, np.abs(hs).max()), dims
        assert np.abs(wg - ws).max() <= tol, dims
