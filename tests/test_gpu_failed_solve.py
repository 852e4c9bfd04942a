"""A groundwater step whose solve fails, as the program finds the fields after the error: a solve that is queued
(whole in one launch) leaves them as one that the host waits for (the streaming solver, pinned by
FREHG_SPMV_SHAPE), although the step's remaining kernels are queued behind it."""
import numpy as np
import pytest

from frehg_amd import abi, gpu
from gpu_common import say

pytestmark = pytest.mark.gpu

FIELDS = ("h", "hn", "wc", "wcn", "wch", "hwc", "ch")


def after_failure(monkeypatch, shape, lazy, picard, guess):
    for name, value in (("FREHG_SPMV_SHAPE", shape), ("FREHG_LAZY_FLUX", lazy)):
        if value is None:
            monkeypatch.delenv(name, raising=False)
        else:
            monkeypatch.setenv(name, value)
    nx, ny, nz = 30, 21, 14
    soil = abi.soil_params(alpha=2.0, n=1.8, theta_s=0.40, theta_r=0.05, Ks_x=1e-5, Ks_y=1e-5, Ks_z=1e-5, Ss=1e-5)

    def params(cfg):
        return abi.re_params(soil=soil, solver=cfg, bc_type=(0, 0, 0, 0, 3, 1), dx=0.5, dy=0.5, dz=0.05, dt=30.0,
                             adaptive_dt=0, use_full3d=1, htop=-0.3, initial_guess=guess, picard_max=picard,
                             picard_tol=1e-8)

    ctx = gpu.Context(0)
    ctx.re_init(nx, ny, nz, params(abi.solver_config(1e-13)))
    rng = np.random.default_rng(4)
    ctx.re_set_initial(h=-1.5 + 0.2 * rng.standard_normal(nx * ny * nz))
    for _ in range(2):
        ctx.re_step()
    ctx.re_set_params(params(abi.solver_config(1e-13, max_it=2)))
    with pytest.raises(gpu.FrehgError) as e:
        ctx.re_step()
    assert e.value.code == abi.ERR_NOT_CONVERGED
    return {f: ctx.re_get(f) for f in FIELDS}


@pytest.mark.parametrize("lazy", [None, "0"])
@pytest.mark.parametrize("picard,guess", [(1, abi.GUESS_ZERO), (1, abi.GUESS_PREVIOUS), (1, abi.GUESS_EXTRAPOLATED),
                                          (30, abi.GUESS_ZERO), (30, abi.GUESS_PREVIOUS)])
def test_failed_queued_solve_leaves_the_fields(monkeypatch, lazy, picard, guess):
    say(f"failed solve: picard {picard} guess {guess} lazy {lazy}")
    a = after_failure(monkeypatch, None, lazy, picard, guess)
    b = after_failure(monkeypatch, "1:1", lazy, picard, guess)
    for f in FIELDS:
        # two solves to 1e-13 before, then two iterations from the same start, in another order of sums; outside
        # of the iterate itself the fields of the failed step's unconverged head differ by far more
        scale = np.abs(b[f]).max()
        assert np.abs(a[f] - b[f]).max() <= 1e-9 * scale, f


@pytest.mark.parametrize("nx,ny", [(40, 45), (150, 97)])  # one block, several
def test_failed_surface_solve_leaves_the_fields(monkeypatch, nx, ny):
    """The same of a surface step, whose kernels behind the solve are queued with it."""
    say(f"failed surface solve: {nx}x{ny}")
    rng = np.random.default_rng(8)
    bed, depth = 0.1 * rng.random((ny, nx)), 0.3 + 0.2 * rng.random((ny, nx))
    fields = []
    for shape in (None, "1:1"):
        if shape:
            monkeypatch.setenv("FREHG_SPMV_SHAPE", shape)
        else:
            monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
        ctx = gpu.Context(0)
        ctx.swe_init(nx, ny, 1.0, 1.0, abi.swe_params(manning=0.03, dt=1.0, solver=abi.solver_config(1e-12, max_it=3)))
        ctx.swe_set_bathymetry(bed.ravel())
        ctx.swe_set_initial_eta((bed + depth).ravel())
        with pytest.raises(gpu.FrehgError) as e:
            ctx.swe_step(1e-5)
        assert e.value.code == abi.ERR_NOT_CONVERGED
        assert (ctx.resident_use()[0] == 1) == (shape is None)
        fields.append({f: ctx.swe_get(f) for f in abi.SWE_FIELDS})
    for f in abi.SWE_FIELDS:
        a, b = (v[f] for v in fields)
        # (three iterations from the same start in another order of sums)
        assert np.abs(a - b).max() <= 1e-9 * max(1.0, np.abs(b).max()), f
