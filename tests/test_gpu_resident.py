"""The resident CG solve (one launch, vectors on the compute units) against the streaming CG on the
same operators: the same iterates up to the order of the sums, so the same iteration counts (within one, at
the tolerance) and solutions to the solver's tolerance. Sizes at the edges of its tilings: one block
(up to 4096 rows), the first sizes with several blocks, 1, 2, 4 and 8 cells per thread, thin
domains whose tiles are limited by their halo, the largest it takes (4096 rows per compute unit) and the
first it does not."""
import numpy as np
import pytest

from frehg_amd import abi, gpu
from gpu_common import say
from test_zz_no_alloc import spd_stencil

pytestmark = pytest.mark.gpu

SIZES = [(3, 1, 1, 7), (3, 1, 1, 853), (3, 1, 1, 900), (3, 13, 9, 7), (3, 16, 16, 16), (3, 17, 16, 16), (3, 3, 2, 800),
         (3, 70, 33, 9), (3, 80, 80, 41), (3, 129, 63, 62), (3, 101, 100, 100), (2, 64, 64, 1), (2, 65, 64, 1),
         (2, 1, 5000, 1), (2, 5000, 1, 1), (2, 363, 362, 1), (2, 1024, 1024, 1), (2, 1025, 1024, 1)]


def solve(monkeypatch, shape, ndim, nx, ny, nz, diag, offs, b, cfg):
    if shape:
        monkeypatch.setenv("FREHG_SPMV_SHAPE", shape)
    else:
        monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
    ctx = gpu.Context(0)
    out = [ctx.ls_solve(ndim, nx, ny, nz, diag, offs, b, cfg) for _ in range(1)][0]
    ctx.close()
    return out


@pytest.mark.parametrize("ndim,nx,ny,nz", SIZES)
@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED])
def test_resident_solve_matches_streaming(monkeypatch, ndim, nx, ny, nz, precision):
    if precision == abi.PREC_MIXED and nx * ny * nz > 600000:
        pytest.skip("one large size per precision is enough")
    say(f"resident CG {ndim}D {nx}x{ny}x{nz} precision {precision}")
    diag, offs, b = spd_stencil(ndim, nx, ny, nz, 11)
    cfg = abi.solver_config(1e-11, precision=precision)
    x, st = solve(monkeypatch, None, ndim, nx, ny, nz, diag, offs, b, cfg)
    xs, ss = solve(monkeypatch, "1:1", ndim, nx, ny, nz, diag, offs, b, cfg)
    assert st.converged and ss.converged and st.iterations > 0
    assert abs(st.iterations - ss.iterations) <= (1 if precision == abi.PREC_FP64 else 4)
    assert st.rhs_norm == pytest.approx(ss.rhs_norm, rel=1e-12)
    # both stop at ||D^-1 r|| <= 1e-11 ||D^-1 b||; cond(D^-1 A) of these operators is below 100
    assert np.linalg.norm(x - xs) <= 2e-9 * np.linalg.norm(xs)


def test_resident_solve_with_fixed_rows_over_several_blocks(monkeypatch):
    """Decoupled (dry) rows, on tile edges among others: solved exactly and left alone."""
    nx, ny = 150, 97
    diag, offs, b = spd_stencil(2, nx, ny, 1, 5)
    rows = np.unique(np.concatenate([np.arange(0, nx * ny, 37), np.arange(20 * nx, 22 * nx)]))
    for d in range(4):
        offs[d] = offs[d].copy()
    for q in rows:
        for d, s in enumerate((-1, 1, -nx, nx)):
            if offs[d][q] != 0.0:
                offs[d ^ 1][q + s] = 0.0
            offs[d][q] = 0.0
    cfg = abi.solver_config(1e-12)
    x, st = solve(monkeypatch, None, 2, nx, ny, 1, diag, offs, b, cfg)
    xs, ss = solve(monkeypatch, "1:1", 2, nx, ny, 1, diag, offs, b, cfg)
    assert np.array_equal(x[rows], b[rows] / diag[rows])
    assert abs(st.iterations - ss.iterations) <= 1
    assert np.linalg.norm(x - xs) <= 1e-9 * np.linalg.norm(xs)


def test_resident_solves_of_two_contexts_in_turn(monkeypatch):
    """Several solves on one instance's exchange buffers, interleaved with another context's."""
    monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
    a, c = gpu.Context(0), gpu.Context(0)
    d1, d2 = spd_stencil(3, 40, 41, 17, 1), spd_stencil(3, 60, 23, 20, 2)
    cfg = abi.solver_config(1e-11)
    first = None
    for _ in range(3):
        x1, _ = a.ls_solve(3, 40, 41, 17, *d1, cfg)
        x2, _ = c.ls_solve(3, 60, 23, 20, *d2, cfg)
        if first is None:
            first = (x1, x2)
        assert np.array_equal(x1, first[0]) and np.array_equal(x2, first[1])


def test_resident_solve_stops_as_the_streaming_one_does():
    ctx = gpu.Context(0)
    diag, offs, b = spd_stencil(3, 30, 30, 30, 3)
    with pytest.raises(gpu.FrehgError) as e:  # max_it
        ctx.ls_solve(3, 30, 30, 30, diag, offs, b, abi.solver_config(1e-14, max_it=2))
    assert e.value.code == abi.ERR_NOT_CONVERGED
    with pytest.raises(gpu.FrehgError) as e:  # p.Ap < 0
        ctx.ls_solve(3, 30, 30, 30, -diag, offs, b, abi.solver_config(1e-10))
    assert "breakdown" in str(e.value)
    x, st = ctx.ls_solve(3, 30, 30, 30, diag, offs, np.zeros_like(b), abi.solver_config(1e-10))
    assert st.iterations == 0 and not x.any()


@pytest.mark.parametrize("precision", [abi.PREC_FP64, abi.PREC_MIXED])
def test_profile_times_the_solves_of_one_launch(monkeypatch, precision):
    """Kernel timing shows the groundwater Krylov work of small grids: whole solves under FREHG_KT_GW_CG, or SpMV
    and update launches where a shape is pinned."""
    nx, ny, nz = 30, 22, 15
    soil = abi.soil_params(alpha=2.0, n=1.8, theta_s=0.40, theta_r=0.05, Ks_x=1e-5, Ks_y=1e-5, Ks_z=1e-5, Ss=1e-5)
    p = abi.re_params(soil=soil, solver=abi.solver_config(1e-11, precision=precision), dx=0.5, dy=0.5, dz=0.05, dt=30.0,
                      bc_type=(0, 0, 0, 0, 3, 1), htop=-0.3, adaptive_dt=0, use_full3d=1)
    for shape in (None, "1:1"):
        if shape:
            monkeypatch.setenv("FREHG_SPMV_SHAPE", shape)
        else:
            monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
        ctx = gpu.Context(0)
        ctx.re_init(nx, ny, nz, p)
        ctx.re_set_initial(h=np.full(nx * ny * nz, -1.5))
        ctx.profile_enable(True)
        ctx.profile_reset()
        solves = 0
        for _ in range(3):
            solves += max(1, ctx.re_step().solve.refinements)
        cg_ms, cg = ctx.profile_read(abi.KT_GW_CG)
        streamed = [ctx.profile_read(kt) for kt in (abi.KT_GW_SPMV, abi.KT_GW_SPMV32, abi.KT_GW_UPDATE)]
        if shape:
            assert cg == 0 and sum(n for _, n in streamed) >= 2 * solves and sum(ms for ms, _ in streamed) > 0.0
        else:
            assert cg == ctx.resident_use()[0] == solves and cg_ms > 0.0 and sum(n for _, n in streamed) == 0
