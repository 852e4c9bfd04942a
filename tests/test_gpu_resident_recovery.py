"""Resident CG launches that give up: forced from the host by FREHG_RESIDENT_WAIT (bounds of 0 for the wait until all
blocks have started, or for the words of blocks that have), and found by two processes that share the device.
Every solve then ends in the streaming kernels with their answer, the work queued behind it is done again, and the
context goes back to one launch after a bounded number of solves."""
import json
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from frehg_amd import abi, gpu, workloads
from gpu_common import say
from test_zz_no_alloc import _solve_noalloc, spd_stencil

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

BOUNDS = ["0:0", "1000000:0"]  # the start gate closed at once; the first wait behind it


@pytest.fixture
def env(monkeypatch):
    for name in ("FREHG_RESIDENT_WAIT", "FREHG_SPMV_SHAPE"):
        monkeypatch.delenv(name, raising=False)
    return monkeypatch


@pytest.mark.parametrize("bounds", BOUNDS)
@pytest.mark.parametrize("ndim,nx,ny,nz", [(3, 13, 16, 20), (3, 80, 80, 41), (3, 128, 96, 48), (2, 90, 70, 1),
                                           (2, 700, 640, 1)])
def test_solves_that_give_up_stream(env, bounds, ndim, nx, ny, nz):
    say(f"resident CG gives up ({bounds}): {ndim}D {nx}x{ny}x{nz}")
    diag, offs, b = spd_stencil(ndim, nx, ny, nz, 3)
    cfg = abi.solver_config(1e-11)
    ctx = gpu.Context(0)
    ref, sref = ctx.ls_solve(ndim, nx, ny, nz, diag, offs, b, cfg)
    n0, g0, _, blocks = ctx.resident_use()
    assert (n0, g0) == (1, 0) and blocks > 1
    env.setenv("FREHG_RESIDENT_WAIT", bounds)
    for solve in (ctx.ls_solve, lambda *a: _solve_noalloc(ctx, *a)):
        tries = ctx.resident_use()[1]
        while ctx.resident_use()[1] == tries:  # past the pause after the last one
            x, st = solve(ndim, nx, ny, nz, diag, offs, b, cfg)
            assert st.converged and abs(st.iterations - sref.iterations) <= 1
            # (both stop at 1e-11 of the right-hand side; cond(D^-1 A) of these operators is below 100)
            assert np.linalg.norm(x - ref) <= 2e-9 * np.linalg.norm(ref)
    n, g = ctx.resident_use()[:2]
    assert n - n0 == g - g0 == 2


def test_the_pause_after_giving_up(env):
    """One try in 1, 2, 4, ... 64 solves more while the device stays shared, and every solve once it is free."""
    diag, offs, b = spd_stencil(3, 40, 30, 20, 8)
    cfg = abi.solver_config(1e-10)
    ctx = gpu.Context(0)
    env.setenv("FREHG_RESIDENT_WAIT", "0:0")
    tries = []
    for k in range(200):
        before = ctx.resident_use()[0]
        _solve_noalloc(ctx, 3, 40, 30, 20, diag, offs, b, cfg)
        if ctx.resident_use()[0] > before:
            tries.append(k)
    assert tries == [0, 2, 5, 10, 19, 36, 69, 134, 199]
    env.delenv("FREHG_RESIDENT_WAIT")
    n, g = ctx.resident_use()[:2]
    for _ in range(64 + 10):
        _solve_noalloc(ctx, 3, 40, 30, 20, diag, offs, b, cfg)
    assert ctx.resident_use()[:2] == (n + 10, g)
    # a solve of one block waits for nobody: it is never paused
    small = spd_stencil(3, 9, 8, 7, 8)
    env.setenv("FREHG_RESIDENT_WAIT", "0:0")
    _solve_noalloc(ctx, 3, 9, 8, 7, *small, cfg)
    assert ctx.resident_use()[:2] == (n + 11, g)


CASES = [(abi.PREC_FP64, abi.GUESS_ZERO, 1), (abi.PREC_FP64, abi.GUESS_PREVIOUS, 1),
         (abi.PREC_FP64, abi.GUESS_ZERO, 40), (abi.PREC_FP64, abi.GUESS_PREVIOUS, 40),
         (abi.PREC_FP64, abi.GUESS_EXTRAPOLATED, 40), (abi.PREC_MIXED, abi.GUESS_ZERO, 1),
         (abi.PREC_MIXED, abi.GUESS_PREVIOUS, 40), (abi.PREC_MIXED, abi.GUESS_EXTRAPOLATED, 40)]


def run_coupled(precision, guess, picard, n=6):
    case = workloads.CoupledCase(nx=70, ny=61, nz=12, rain=5e-4)
    ctx = gpu.Context(0)
    case.setup_gpu(ctx, precision, guess, picard_max=picard)
    stats = [ctx.coupled_step(case.cp, case.dt, case.rain, 0.0, case.t_end) for _ in range(n)]
    return ctx, stats


@pytest.mark.parametrize("bounds", BOUNDS)
@pytest.mark.parametrize("precision,guess,picard", CASES)
def test_coupled_steps_whose_solves_give_up(env, bounds, precision, guess, picard):
    """Surface and groundwater steps with the kernels queued behind the solve done again, every field against the
    run whose launches complete."""
    say(f"coupled 70x61x12 gives up ({bounds}): precision {precision} guess {guess} picard {picard}")
    ref, sr = run_coupled(precision, guess, picard)
    assert ref.resident_use()[1] == 0 and ref.resident_use()[0] > 0
    env.setenv("FREHG_RESIDENT_WAIT", bounds)
    ctx, st = run_coupled(precision, guess, picard)
    n, g = ctx.resident_use()[:2]
    # (behind the gate, a solve that converges at its first sums waits for nothing more)
    assert g == n >= 3 if bounds == "0:0" else 2 <= g <= n
    # each solve ends at 1e-10 or below of its right-hand side in both runs, and the Picard iterates at 1e-8 m
    tol = 1e-7 if picard > 1 or precision == abi.PREC_MIXED else 1e-8
    for f in ("h", "hn", "wc", "wcn", "wch"):
        a, b = ctx.re_get(f), ref.re_get(f)
        assert np.abs(a - b).max() <= tol * max(1.0, np.abs(b).max()), f
    for f in ("eta", "etan", "dept", "uu", "vv", "un", "vn", "Vs", "Vsn"):
        a, b = ctx.swe_get(f), ref.swe_get(f)
        assert np.abs(a - b).max() <= tol * max(1.0, np.abs(b).max()), f
    for a, b in zip(st, sr):
        assert a.gw.solve.converged and (picard == 1 or a.gw.picard_converged)
        assert abs(a.gw.picard_iterations - b.gw.picard_iterations) <= 1


CHILD = """
import json, sys, time
import numpy as np
sys.path[:0] = [{root!r}]
from frehg_amd import abi, gpu, workloads
case = workloads.CoupledCase(nx=128, ny=120, nz=30)
ctx = gpu.Context(0)
case.setup_gpu(ctx, abi.PREC_FP64, abi.GUESS_ZERO)
ctx.coupled_step(case.cp, case.dt, case.rain, 0.0, case.t_end)
print("ready", flush=True)
sys.stdin.readline()
t0 = time.time()
for _ in range(400):
    ctx.coupled_step(case.cp, case.dt, case.rain, 0.0, case.t_end)
dt = time.time() - t0
np.savez(sys.argv[1], h=ctx.re_get("h"), eta=ctx.swe_get("eta"))
print(json.dumps(dict(seconds=dt, use=ctx.resident_use())), flush=True)
"""


def processes(tmp_path, n):
    child = tmp_path / "child.py"
    child.write_text(CHILD.format(root=ROOT))
    outs = [str(tmp_path / f"out{n}_{k}.npz") for k in range(n)]
    ps = [subprocess.Popen([sys.executable, str(child), o], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
          for o in outs]
    watchdog = threading.Timer(90.0, lambda: [p.kill() for p in ps])  # (a read below has no time limit of its own)
    watchdog.start()
    try:
        for p in ps:
            assert p.stdout.readline().strip() == "ready"
        for p in ps:
            p.stdin.write("\n")
            p.stdin.flush()
        res = [json.loads(p.communicate(timeout=60)[0].splitlines()[-1]) for p in ps]
    finally:
        watchdog.cancel()
        for p in ps:
            if p.poll() is None:
                p.kill()
            p.wait()
    return res, [np.load(o) for o in outs]


def test_two_processes_share_the_device(env, tmp_path):
    """Solves of more than 128 blocks from two processes at once: together they do not fit on the 256 compute units.
    Each run ends with the result of the run alone, without a wait of a quarter of a second per solve."""
    say("two processes, 128x120x30")
    (alone,), (ref,) = processes(tmp_path, 1)
    say(f"alone: {alone}")
    assert alone["use"][1] == 0 and alone["use"][3] > 128
    both, outs = processes(tmp_path, 2)
    say(f"two: {both}")
    for r, o in zip(both, outs):
        for f in ("h", "eta"):
            assert np.abs(o[f] - ref[f]).max() <= 1e-8 * max(1.0, np.abs(ref[f]).max()), f
        # at most 5 ms per launch that gave up, and a streamed step takes some ms here
        assert r["seconds"] < 10.0, both
