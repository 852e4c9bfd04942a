"""The resident CG solve (one launch, vectors on the compute units) against the streaming CG on the
same operators: the same iterates up to the order of the sums, so the same iteration counts (within one, at
the tolerance) and solutions to the solver's tolerance. Sizes at the edges of its tilings, which each test
checks were the ones that ran: one block (up to 2048 rows) with 1, 2 and 4 cells per thread and the first sizes
with several, several blocks with 1, 2, 4 and 8, thin domains whose tiles are limited by their halo, the largest
that run in one launch (2D: 4096 rows per compute unit; 3D in FP64: what fits the LDS with the operator) and the
first that do not. The FP32 kernel, started by a refinement sweep, runs in mixed-precision Richards steps."""
import numpy as np
import pytest

from frehg_amd import abi, gpu
from gpu_common import say
from test_zz_no_alloc import spd_stencil

pytestmark = pytest.mark.gpu

# (ndim, nx, ny, nz), cells per thread (0: streams) and blocks on 256 compute units
SIZES = [((3, 1, 1, 7), 1, 1), ((3, 1, 1, 853), 2, 1), ((3, 1, 1, 900), 1, 2), ((3, 13, 9, 7), 2, 1),
         ((3, 5, 5, 41), 4, 1), ((3, 13, 12, 13), 4, 1), ((3, 11, 11, 17), 1, 36), ((3, 16, 16, 16), 1, 64),
         ((3, 17, 16, 16), 1, 48), ((3, 3, 2, 800), 1, 10), ((3, 70, 33, 9), 1, 70), ((3, 80, 70, 40), 2, None),
         ((3, 80, 80, 41), 4, 192), ((3, 129, 63, 62), 4, 252), ((3, 128, 96, 48), 8, 240), ((3, 127, 95, 47), 8, 240),
         ((3, 100, 90, 90), 8, 252), ((3, 101, 100, 100), 0, 0), ((2, 45, 45, 1), 4, 1), ((2, 46, 45, 1), 1, 12),
         ((2, 64, 64, 1), 1, 16), ((2, 65, 64, 1), 1, None), ((2, 1, 5000, 1), 1, 65), ((2, 5000, 1, 1), 1, 65),
         ((2, 363, 362, 1), 2, 132), ((2, 600, 600, 1), 4, 180), ((2, 1024, 1024, 1), 8, 256), ((2, 1025, 1024, 1), 0, 0)]


def solve(monkeypatch, shape, ndim, nx, ny, nz, diag, offs, b, cfg):
    if shape:
        monkeypatch.setenv("FREHG_SPMV_SHAPE", shape)
    else:
        monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
    ctx = gpu.Context(0)
    out = ctx.ls_solve(ndim, nx, ny, nz, diag, offs, b, cfg)
    use = ctx.resident_use()
    ctx.close()
    return (*out, use)


@pytest.mark.parametrize("size,cells,blocks", SIZES)
def test_resident_solve_matches_streaming(monkeypatch, size, cells, blocks):
    ndim, nx, ny, nz = size
    say(f"resident CG {ndim}D {nx}x{ny}x{nz}")
    diag, offs, b = spd_stencil(ndim, nx, ny, nz, 11)
    cfg = abi.solver_config(1e-11)
    x, st, use = solve(monkeypatch, None, ndim, nx, ny, nz, diag, offs, b, cfg)
    xs, ss, none = solve(monkeypatch, "1:1", ndim, nx, ny, nz, diag, offs, b, cfg)
    launches, gave_up, cpt, nblk = use
    assert (launches, gave_up, cpt) == ((1, 0, cells) if cells else (0, 0, 0)) and none[0] == 0
    assert blocks is None or nblk == blocks
    assert st.converged and ss.converged and st.iterations > 0
    assert abs(st.iterations - ss.iterations) <= 1
    assert st.rhs_norm == pytest.approx(ss.rhs_norm, rel=1e-12)
    # both stop at ||D^-1 r|| <= 1e-11 ||D^-1 b||; cond(D^-1 A) of these operators is below 100
    assert np.linalg.norm(x - xs) <= 2e-9 * np.linalg.norm(xs)


# FP32 inner solves: (nx, ny, nz), cells per thread, whether several blocks
MIXED = [((6, 6, 10), 1, False), ((13, 9, 7), 2, False), ((16, 16, 8), 4, False), ((1, 1, 900), 2, False),
         ((30, 30, 30), 1, True), ((80, 70, 40), 2, True), ((100, 80, 64), 4, True), ((128, 96, 48), 8, True),
         ((101, 100, 100), 8, True)]


@pytest.mark.parametrize("size,cells,several", MIXED)
@pytest.mark.parametrize("guess,picard", [(abi.GUESS_ZERO, 1), (abi.GUESS_PREVIOUS, 30)])
def test_mixed_precision_steps_match_streaming(monkeypatch, size, cells, several, guess, picard):
    nx, ny, nz = size
    say(f"resident FP32 CG {nx}x{ny}x{nz} guess {guess} picard {picard}")
    soil = abi.soil_params(alpha=2.0, n=1.8, theta_s=0.40, theta_r=0.05, Ks_x=1e-5, Ks_y=1e-5, Ks_z=1e-5, Ss=1e-5)
    p = abi.re_params(soil=soil, solver=abi.solver_config(1e-11, precision=abi.PREC_MIXED), dx=0.5, dy=0.5, dz=0.05,
                      dt=30.0, bc_type=(0, 0, 0, 0, 3, 1), htop=-0.3, adaptive_dt=0, use_full3d=1,
                      initial_guess=guess, picard_max=picard, picard_tol=1e-8)
    h0 = -1.5 + 0.2 * np.random.default_rng(3).standard_normal(nx * ny * nz)
    heads, stats = [], []
    for shape in (None, "1:1"):
        if shape:
            monkeypatch.setenv("FREHG_SPMV_SHAPE", shape)
        else:
            monkeypatch.delenv("FREHG_SPMV_SHAPE", raising=False)
        ctx = gpu.Context(0)
        ctx.re_init(nx, ny, nz, p)
        ctx.re_set_initial(h=h0)
        stats.append([ctx.re_step() for _ in range(3)])
        heads.append(ctx.re_get("h"))
        launches, gave_up, cpt, blocks = ctx.resident_use()
        if shape:
            assert launches == 0
        else:
            assert launches >= 3 and gave_up == 0 and cpt == cells and (blocks > 1) == several
        ctx.close()
    for a, b in zip(*stats):
        assert a.solve.converged and b.solve.converged and a.solve.fallback == b.solve.fallback == 0
        assert a.picard_iterations == b.picard_iterations and a.picard_converged == b.picard_converged
    # each solve ends at 1e-11 of its right-hand side (heads of a few metres), Picard iterates at 1e-8 m
    assert np.abs(heads[0] - heads[1]).max() <= (1e-8 if picard == 1 else 1e-7)


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
    x, st, use = solve(monkeypatch, None, 2, nx, ny, 1, diag, offs, b, cfg)
    xs, ss, _ = solve(monkeypatch, "1:1", 2, nx, ny, 1, diag, offs, b, cfg)
    assert use[0] == 1 and use[1] == 0 and use[3] > 1
    assert np.array_equal(x[rows], b[rows] / diag[rows])
    assert abs(st.iterations - ss.iterations) <= 1
    assert np.linalg.norm(x - xs) <= 1e-9 * np.linalg.norm(xs)


def test_resident_solves_of_two_contexts_in_turn(monkeypatch):
    """Single solves (each with a solver and exchange buffers of its own) on two contexts in turn: the same bits every
    time. (Solvers that live on, and several threads: test_gpu_two_contexts.py.)"""
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
    assert a.resident_use()[:2] == c.resident_use()[:2] == (3, 0)


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
