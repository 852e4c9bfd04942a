"""The work that is timed: what a program built on this framework has it do, through the package's
public entry points (frehg_amd.gpu, which binds include/frehg_gpu.h), over the sizes it is used at.

Kinds of case ("kind" of a case):

  solve     one call of the linear solver seam on device arrays (frehg_ls_solve_noalloc): a program that
            keeps its own assembly and replaces only the Krylov solve.
  re        groundwater only: an infiltration run, from its initial state to its next output.
  ensemble  a batch of independent groundwater boxes of uneven size, advanced to its next output.
  swe       surface only: a basin advanced to its next output.
  coupled   the coupled surface / groundwater model advanced to its next output, with the solver
            settings of the YAML front end's defaults (FP64, zero start, one iterate per step) or of
            the Picard method with the mixed-precision solver and the extrapolated or learned start.
  mlp       the learned start's network: loss and gradient of a batch, and its predictions.

One pass is the time steps between two outputs and the read-back of the state that an output writes,
into pinned host memory that the program keeps. The coupled, ensemble and larger surface cases go on
from where the last pass ended, as a simulation does: a storm of 300 s falls on the coupled ones, then the
water redistributes. The small ones start again from their initial state in every pass.
"""
import ctypes as C
import math

import numpy as np
import torch

from frehg_amd import abi, gpu

DEV = "cuda"
STORM = 300.0  # s: rain falls until then

GUESS = {"zero": abi.GUESS_ZERO, "previous": abi.GUESS_PREVIOUS, "learned": abi.GUESS_LEARNED,
         "extrapolated": abi.GUESS_EXTRAPOLATED}


def listed():
    return [
        # The smallest solve: a test-sized operator, all launches and round trips.
        {"name": "solve3d_13x9x7", "kind": "solve", "ndim": 3, "nx": 13, "ny": 9, "nz": 7, "dt": 1.0, "rtol": 1e-10},
        # A solve near the largest that the allocation-free entry takes, groundwater couplings.
        {"name": "solve3d_128x96x48", "kind": "solve", "ndim": 3, "nx": 128, "ny": 96, "nz": 48, "dt": 30.0,
         "rtol": 1e-10},
        # A single soil column under a ponded top with adaptive dt (the b2-gw benchmark's set-up).
        {"name": "column_1x1x100_adaptive", "kind": "re", "nx": 1, "ny": 1, "nz": 100, "set": "column", "steps": 30,
         "precision": "fp64", "guess": "zero", "picard": 1, "ksp": "cg", "soil": "uniform"},
        # The 40x40x50 infiltration benchmark: Picard to 1e-8 m in FP64, dt 10 s, free drainage.
        {"name": "infiltration_40x40x50", "kind": "re", "nx": 40, "ny": 40, "nz": 50, "set": "infiltration",
         "steps": 20, "precision": "fp64", "guess": "zero", "picard": 50, "ksp": "cg", "soil": "uniform"},
        # A small catchment's surface water, rain on wet and dry ground.
        {"name": "surface_40x60_wetdry", "kind": "swe", "nx": 40, "ny": 60, "wet": False, "steps": 20, "ksp": "cg"},
        # A large basin, all wet: waves over a random bed.
        {"name": "surface_512x512_wet", "kind": "swe", "nx": 512, "ny": 512, "wet": True, "steps": 20, "ksp": "cg"},
        # The coupled benchmark with the front end's default solver settings (the reference's step).
        {"name": "coupled_512x512x30_predictor", "kind": "coupled", "nx": 512, "ny": 512, "nz": 30, "steps": 10,
         "precision": "fp64", "guess": "zero", "picard": 1, "solute": False, "large": False},
        # The coupled benchmark as the framework runs it fastest: Picard, mixed precision, learned start.
        {"name": "coupled_512x512x30_learned", "kind": "coupled", "nx": 512, "ny": 512, "nz": 30, "steps": 10,
         "precision": "mixed", "guess": "learned", "picard": 50, "solute": False, "large": False},
        # A ragged catchment with a tracer: odd sizes, Picard in FP64 from the previous head.
        {"name": "coupled_201x157x23_solute", "kind": "coupled", "nx": 201, "ny": 157, "nz": 23, "steps": 10,
         "precision": "fp64", "guess": "previous", "picard": 50, "solute": True, "large": False},
        # The largest configuration: 67 million soil cells, Picard, mixed precision, extrapolated start.
        {"name": "coupled_1024x1024x64", "kind": "coupled", "nx": 1024, "ny": 1024, "nz": 64, "steps": 4,
         "precision": "mixed", "guess": "extrapolated", "picard": 50, "solute": False, "large": True},
        # A batch of uneven boxes (a parameter study), replayed from captured graphs.
        {"name": "ensemble_24_boxes", "kind": "ensemble", "boxes": 24, "lo": 32, "hi": 128, "steps": 3,
         "precision": "mixed", "guess": "extrapolated"},
        # One minibatch of the learned start's training: loss, gradient and predictions.
        {"name": "network_65536", "kind": "mlp", "batch": 65536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "re", "re", "swe", "coupled", "coupled", "coupled", "ensemble", "mlp"])
    if kind == "solve":
        if rng.random() < 0.5:
            return {"kind": kind, "ndim": 2, "nx": _log(rng, 8, 600), "ny": _log(rng, 8, 600), "nz": 1,
                    "dt": round(rng.uniform(0.5, 2.0), 3), "rtol": 1e-12}
        return {"kind": kind, "ndim": 3, "nx": _log(rng, 4, 128), "ny": _log(rng, 4, 96), "nz": _log(rng, 3, 48),
                "dt": round(math.exp(rng.uniform(0.0, math.log(60.0))), 3), "rtol": 1e-10}
    if kind == "re":
        if rng.random() < 0.3:
            return {"kind": kind, "nx": 1, "ny": 1, "nz": _log(rng, 40, 200), "set": "column",
                    "steps": rng.randint(10, 40), "precision": "fp64", "guess": "zero", "picard": 1,
                    "ksp": rng.choice(["cg", "cg", "bcgs"]), "soil": "uniform"}
        return {"kind": kind, "nx": _log(rng, 9, 180), "ny": _log(rng, 9, 180), "nz": _log(rng, 10, 90),
                "set": "infiltration", "steps": rng.randint(5, 15), "precision": rng.choice(["fp64", "mixed"]),
                "guess": rng.choice(["zero", "previous", "extrapolated"]), "picard": rng.choice([1, 50]),
                "ksp": rng.choice(["cg", "cg", "bcgs"]), "soil": rng.choice(["uniform", "ks", "classes"])}
    if kind == "swe":
        return {"kind": kind, "nx": _log(rng, 16, 700), "ny": _log(rng, 16, 700), "wet": rng.random() < 0.5,
                "steps": rng.randint(10, 30), "ksp": "cg"}
    if kind == "ensemble":
        return {"kind": kind, "boxes": rng.randint(3, 24), "lo": 17, "hi": rng.randint(48, 120), "steps": 3,
                "precision": rng.choice(["fp64", "mixed"]), "guess": rng.choice(["zero", "previous", "extrapolated"])}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 500, 200000)}
    guess, precision = rng.choice([("zero", "fp64"), ("previous", "fp64"), ("previous", "mixed"),
                                   ("extrapolated", "mixed"), ("learned", "mixed")])
    return {"kind": kind, "nx": _log(rng, 24, 600), "ny": _log(rng, 24, 600), "nz": _log(rng, 8, 40),
            "steps": rng.randint(5, 10), "precision": precision, "guess": guess,
            "picard": 50 if guess == "learned" else rng.choice([1, 50]), "solute": rng.random() < 0.25, "large": False}


# ---- inputs -------------------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * (int(seed) % (1 << 40)) + salt)


def _grf(shape, spacing, corr, sigma, g):
    """Zero-mean Gaussian random field with covariance sigma^2 exp(-r^2 / corr^2) (periodic, by FFT)."""
    f = torch.fft.rfftn(torch.randn(shape, generator=g, device=DEV, dtype=torch.float64))
    for a, (n, d) in enumerate(zip(shape, spacing)):
        fr = torch.fft.rfftfreq(n, d=d, device=DEV, dtype=torch.float64) if a == len(shape) - 1 else \
            torch.fft.fftfreq(n, d=d, device=DEV, dtype=torch.float64)
        v = [1] * len(shape)
        v[a] = -1
        f = f * torch.exp(-(2 * math.pi * fr) ** 2 * corr ** 2 / 8).reshape(v)
    out = torch.fft.irfftn(f, s=shape)
    out = out - out.mean()
    sd = out.std()
    return sigma * out / sd if float(sd) > 0 else out


def _solver(c, rtol):
    return abi.solver_config(rtol, precision=abi.PREC_MIXED if c.get("precision") == "mixed" else abi.PREC_FP64,
                             ksp_type=abi.KSP_BICGSTAB if c.get("ksp") == "bcgs" else abi.KSP_CG)


class _Mirror:
    """Host mirrors of device fields that the program keeps: pinned, packed halo-padded layout."""

    def __init__(self, shape):
        self.keep = torch.empty([n + 2 for n in shape], dtype=torch.float64, pin_memory=True)
        self.a = self.keep.numpy()
        self.ptr = self.a.ctypes.data_as(C.POINTER(C.c_double))
        self.inner = self.a[tuple(slice(1, -1) for _ in shape)]


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(s):
    return s["run"](s)


def _operator(c, seed):
    """Groundwater-like (3D) or surface-like (2D) symmetric operator in the owned row order, with the
    right-hand side of a smooth head: dict of device tensors."""
    g = _gen(seed, 1)
    nx, ny, nz, dt = c["nx"], c["ny"], c["nz"], c["dt"]
    if c["ndim"] == 3:  # rows (j, i, k), k fastest
        K = 2e-6 * torch.exp(_grf((ny, nx, nz), (1.0, 1.0, 0.05), 10.0, 1.0, g))
        V, cap = 0.05, 0.05
        off = {}
        for d, (ax, fac) in enumerate(((1, dt * 0.05), (0, dt * 0.05), (2, dt / 0.05))):
            lo = [slice(None)] * 3
            hi = [slice(None)] * 3
            lo[ax], hi[ax] = slice(0, -1), slice(1, None)
            f = -fac * 0.5 * (K[tuple(lo)] + K[tuple(hi)])
            p, m = torch.zeros_like(K), torch.zeros_like(K)
            p[tuple(lo)] = f
            m[tuple(hi)] = f
            off[2 * d], off[2 * d + 1] = m, p
        D = cap * V * (0.5 + torch.rand(K.shape, generator=g, device=DEV, dtype=torch.float64))
        h = -2.0 + _grf((ny, nx, nz), (1.0, 1.0, 0.05), 10.0, 0.5, g)
    else:  # rows (j, i), i fastest; area + g dt^2 depth per face
        dep = 0.05 + 0.5 * torch.rand((ny, nx), generator=g, device=DEV, dtype=torch.float64)
        off = {}
        for d, ax in enumerate((1, 0)):
            lo = [slice(None)] * 2
            hi = [slice(None)] * 2
            lo[ax], hi[ax] = slice(0, -1), slice(1, None)
            f = -9.81 * dt * dt * 0.5 * (dep[tuple(lo)] + dep[tuple(hi)])
            p, m = torch.zeros_like(dep), torch.zeros_like(dep)
            p[tuple(lo)] = f
            m[tuple(hi)] = f
            off[2 * d], off[2 * d + 1] = m, p
        D = torch.ones_like(dep)
        h = 1.0 + 0.2 * torch.randn((ny, nx), generator=g, device=DEV, dtype=torch.float64)
    for a in off.values():
        D = D - a
    op = {"D": D.contiguous(), "off": [off[d].contiguous() for d in range(2 * c["ndim"])], "ndim": c["ndim"]}
    op["b"] = _apply(op, h).contiguous()
    return op


def _apply(op, x):
    y = op["D"] * x
    axes = (1, 0, 2)[:op["ndim"]]
    for d, ax in enumerate(axes):
        lo = [slice(None)] * op["ndim"]
        hi = [slice(None)] * op["ndim"]
        lo[ax], hi[ax] = slice(0, -1), slice(1, None)
        y[tuple(hi)] += op["off"][2 * d][tuple(hi)] * x[tuple(lo)]
        y[tuple(lo)] += op["off"][2 * d + 1][tuple(lo)] * x[tuple(hi)]
    return y


def _cg(op, b, tol=1e-14, most=3000):
    x = torch.zeros_like(b)
    r, z = b.clone(), b / op["D"]
    p, rz, stop = z.clone(), (b * (b / op["D"])).sum(), tol * float((b / op["D"]).norm())
    for _ in range(most):
        if float(z.norm()) <= stop:
            break
        q = _apply(op, p)
        a = rz / (p * q).sum()
        x, r = x + a * p, r - a * q
        z = r / op["D"]
        new = (r * z).sum()
        p, rz = z + (new / rz) * p, new
    return x


def _prepare_solve(c, seed):
    op = _operator(c, seed)
    x = torch.empty_like(op["b"])
    ctx = gpu.Context(0)
    torch.cuda.synchronize()
    args = (c["ndim"], c["nx"], c["ny"], c["nz"], op["D"].data_ptr(), [o.data_ptr() for o in op["off"]],
            op["b"].data_ptr(), x.data_ptr(), abi.solver_config(c["rtol"]))
    return {"run": _run_solve, "ctx": ctx, "args": args, "op": op, "x": x}


def _run_solve(s):
    s["ctx"].ls_solve_noalloc(*s["args"])
    return s["x"]


def _soils(c, seed):
    """Classes, class index and per-cell Ks of a groundwater case."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    if c["set"] == "column":
        return [abi.soil_params(alpha=1.43, n=1.56, theta_s=0.33, Ks_z=2.89e-6, Ss=1e-5)], None, None
    base = dict(alpha=3.35, n=2.0, theta_s=0.368, theta_r=0.102, Ss=1e-6)
    one = abi.soil_params(Ks_x=9.22e-5, Ks_y=9.22e-5, Ks_z=9.22e-5, **base)
    g = _gen(seed, 2)
    if c["soil"] == "ks":
        return [one], None, (9.22e-5 * torch.exp(_grf((nz, ny, nx), (0.02, 0.1, 0.1), 0.5, 0.5, g))).cpu().numpy()
    if c["soil"] == "classes":
        two = abi.soil_params(alpha=2.0, n=1.6, theta_s=0.42, theta_r=0.06, Ks_x=2e-5, Ks_y=2e-5, Ks_z=2e-5, Ss=1e-6)
        idx = (_grf((nz, ny, nx), (0.02, 0.1, 0.1), 0.5, 1.0, g) > 0.3).to(torch.int32).cpu().numpy()
        return [one, two], idx, None
    return [one], None, None


def _re_setup(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    soils, idx, ks = _soils(c, seed)
    g = _gen(seed, 3)
    kw = dict(soil=soils[0], picard_max=c["picard"], initial_guess=GUESS[c["guess"]], use_full3d=1)
    if c["set"] == "column":
        p = abi.re_params(solver=_solver(c, 1e-12), bc_type=(0, 0, 0, 0, 0, 1), dz=0.01, dt=1e-4, htop=0.0, **kw)
        wc = 0.033 + 0.02 * torch.rand((nz, ny, nx), generator=g, device=DEV, dtype=torch.float64)
        return p, soils, idx, ks, None, wc.cpu().numpy()
    p = abi.re_params(solver=_solver(c, 1e-10), bc_type=(0, 0, 0, 0, 3, 1), dx=0.1, dy=0.1, dz=0.02, botz=-0.02 * nz,
                      dt=10.0, adaptive_dt=0, htop=-0.75, **kw)
    h = -10.0 + _grf((nz, ny, nx), (0.02, 0.1, 0.1), 0.5, 0.3, g)
    return p, soils, idx, ks, h.cpu().numpy(), None


def _prepare_re(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    p, soils, idx, ks, h, wc = _re_setup(c, seed)
    ctx = gpu.Context(0)
    ctx.re_init(nx, ny, nz, p)
    if len(soils) > 1 or ks is not None:
        ctx.re_set_soil(soils, idx, idx is not None, ks)
    return {"run": _run_re, "ctx": ctx, "case": c, "dt": p.dt, "h": h, "wc": wc, "out": [_Mirror((nz, ny, nx)) for _ in range(2)]}


def _read(ctx, fn, names, mirrors):
    for nm, m in zip(names, mirrors):
        ctx.check(fn(ctx.h, nm, m.ptr))


def _run_re(s):
    ctx = s["ctx"]
    ctx.check(ctx.lib.frehg_re_prime_dt(ctx.h, s["dt"]))
    ctx.re_set_initial(h=s["h"], wc=s["wc"])
    for _ in range(s["case"]["steps"]):
        ctx.re_step()
    _read(ctx, ctx.lib.frehg_re_get_field, (b"h", b"wc"), s["out"])
    return {"h": s["out"][0].inner, "wc": s["out"][1].inner, "dt": ctx.re_dt()}


def _boxes(c, seed):
    rng = np.random.Generator(np.random.Philox(int(seed) % (1 << 40)))
    shape = np.random.Generator(np.random.Philox(3))  # the boxes of one study keep their sizes
    boxes = []
    for b in range(c["boxes"]):
        nx, ny = (int(v) for v in shape.integers(c["lo"], c["hi"] + 1, size=2))
        nz = int(shape.integers(20, 121))
        soil = abi.soil_params(alpha=float(rng.uniform(0.5, 5.0)), n=float(rng.uniform(1.3, 2.8)), theta_s=0.40,
                               theta_r=0.05, Ks_x=1e-5, Ks_y=1e-5, Ks_z=1e-5, Ss=1e-5)
        ks = 1e-5 * torch.exp(_grf((nz, ny, nx), (0.05, 0.5, 0.5), 2.0, 1.0, _gen(seed, 100 + b)))
        p = abi.re_params(soil=soil, solver=_solver(c, 1e-10), bc_type=(0, 0, 0, 0, 0, 2), dx=0.5, dy=0.5, dz=0.05,
                          botz=-0.05 * nz, dt=30.0, adaptive_dt=0, use_full3d=1, qtop=-1e-6,
                          initial_guess=GUESS[c["guess"]])
        boxes.append((nx, ny, nz, p, soil, ks.cpu().numpy(), float(rng.uniform(-5.0, -0.5))))
    return boxes


def _prepare_ensemble(c, seed):
    boxes = _boxes(c, seed)
    ctx = gpu.Context(0)
    ctx.ens_init([b[:3] for b in boxes], [b[3] for b in boxes])
    for i, (nx, ny, nz, _, soil, ks, h0) in enumerate(boxes):
        ctx.ens_set_soil(i, [soil], None, True, ks)
        ctx.ens_set_initial(i, h=np.full(nx * ny * nz, h0))
    return {"run": _run_ensemble, "ctx": ctx, "case": c, "out": [_Mirror((b[2], b[1], b[0])) for b in boxes]}


def _run_ensemble(s):
    ctx = s["ctx"]
    for _ in range(s["case"]["steps"]):
        ctx.ens_step(use_graph=True)
    for i, m in enumerate(s["out"]):
        ctx.check(ctx.lib.frehg_ens_get_field(ctx.h, i, b"h", m.ptr))
    return [m.inner for m in s["out"]]


def _prepare_swe(c, seed):
    nx, ny = c["nx"], c["ny"]
    g = _gen(seed, 4)
    x = torch.arange(nx, device=DEV, dtype=torch.float64) + 0.5
    bed = 0.01 * x[None, :] + _grf((ny, nx), (1.0, 1.0), 20.0, 0.05, g)
    if c["wet"]:  # a basin about a metre deep, with waves
        bed = bed - 0.01 * x[None, :]
        eta, rain = 1.0 + _grf((ny, nx), (1.0, 1.0), 30.0, 0.02, g), 0.0
    else:  # ponds in the lower half of a tilted catchment, dry above, rain everywhere
        eta, rain = torch.full_like(bed, float(bed.mean())), 50e-3 / 3600.0
    bed, eta = bed.cpu().numpy(), eta.cpu().numpy()
    ctx = gpu.Context(0)
    p = abi.swe_params(solver=_solver(c, 1e-12), manning=0.03, dt=0.5, offset=-float(bed.min()))
    ctx.swe_init(nx, ny, 1.0, 1.0, p)
    ctx.swe_set_bathymetry(bed + p.offset)
    ctx.swe_set_initial_eta(eta)
    return {"run": _run_swe, "ctx": ctx, "case": c, "eta": eta, "rain": rain, "out": [_Mirror((ny, nx)) for _ in range(3)]}


def _run_swe(s):
    ctx = s["ctx"]
    if not s["case"]["wet"]:
        ctx.swe_set_initial_eta(s["eta"])
    for _ in range(s["case"]["steps"]):
        ctx.swe_step(s["rain"])
    _read(ctx, ctx.lib.frehg_swe_get_field, (b"eta", b"uu", b"vv"), s["out"])
    return {"eta": s["out"][0].inner, "uu": s["out"][1].inner, "vv": s["out"][2].inner}


def _coupled_context(c, seed, nx, ny, nz, precision, guess, picard):
    """A coupled context of the benchmark's recipe: a tilted plane with a random bed, lognormal Ks, a
    critical-depth outflow on the low-x edge, closed sides and bottom, initial head -2 m."""
    dx, dz = (2.0, 0.04) if c["large"] else (1.0, 0.05)
    x = (torch.arange(nx, device=DEV, dtype=torch.float64) + 0.5) * dx
    bed = (0.01 * x[None, :] + _grf((ny, nx), (dx, dx), 20.0, 0.05, _gen(seed, 5))).cpu().numpy()
    ks = (1e-5 * torch.exp(_grf((nz, ny, nx), (dz, dx, dx), 10.0, 1.0, _gen(seed, 6)))).cpu().numpy()
    soil = abi.soil_params(alpha=2.0, n=1.8, theta_s=0.40, theta_r=0.05, Ks_x=1e-5, Ks_y=1e-5, Ks_z=1e-5, Ss=1e-5)
    sp = abi.swe_params(manning=0.03, dt=1.0, offset=-float(bed.min()))
    rp = abi.re_params(soil=soil, solver=_solver({"precision": precision}, 1e-10), bc_type=(0,) * 6, dx=dx, dy=dx, dz=dz,
                       botz=-dz * nz, dt=1.0, adaptive_dt=0, use_full3d=1, initial_guess=guess, picard_max=picard)
    ctx = gpu.Context(0)
    ctx.swe_init(nx, ny, dx, dx, sp)
    ctx.swe_set_bathymetry(bed + sp.offset)
    ctx.swe_initialize_state(-1.0e3)  # dry
    ly = ny * dx
    ctx.swe_set_boundary_polygons([(abi.BC_CRITICAL, 0.0, [(-dx, -dx), (dx, -dx), (dx, ly + dx), (-dx, ly + dx)])])
    ctx.re_init(nx, ny, nz, rp)
    ctx.re_set_soil([soil], None, True, ks)
    ctx.re_set_initial(h=np.full(nx * ny * nz, -2.0))
    return ctx, abi.coupling_params(dx=dx, dy=dx)


def _rain(t):
    return 50e-3 / 3600.0 if t < STORM else 0.0


def _network(c, seed):
    """Weights trained on the first steps of another, smaller realisation of the same recipe."""
    nx = ny = 160
    nz = min(c["nz"], 30)
    ctx, cp = _coupled_context(c, seed, nx, ny, nz, "fp64", abi.GUESS_ZERO, 50)
    ctx.mlp_init(17)
    ctx.mlp_log(4, 10 * (nx * ny * nz // 4 + 1))
    for _ in range(11):
        ctx.coupled_step(cp, 1.0, _rain(0.0), 0.0, 1800.0)
    ctx.mlp_train(1000, batch=65536, lr=1e-3, seed=29)
    model = ctx.mlp_get_params()
    ctx.close()
    return model


def _prepare_coupled(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    model = _network(c, seed + 7919) if c["guess"] == "learned" else None
    ctx, cp = _coupled_context(c, seed, nx, ny, nz, c["precision"], GUESS[c["guess"]], c["picard"])
    if model is not None:
        ctx.mlp_set_params(*model)
        ctx.mlp_gate(1e-6)
    out = [_Mirror((nz, ny, nx)), _Mirror((nz, ny, nx)), _Mirror((ny, nx))]
    if c["solute"]:
        ctx.solute_init(abi.solute_params(muscl=1, D=1e-9, c_rain=0.1))
        patch = np.zeros((ny, nx))
        patch[ny // 4:ny // 2 + 1, nx // 4:nx // 2 + 1] = 1.0
        ctx.solute_set_initial(patch, None)
        out += [_Mirror((ny, nx)), _Mirror((nz, ny, nx))]
    return {"run": _run_coupled, "ctx": ctx, "case": c, "cp": cp, "t": 0.0, "out": out}


def _run_coupled(s):
    ctx, c, out = s["ctx"], s["case"], s["out"]
    for _ in range(c["steps"]):
        ctx.coupled_step(s["cp"], 1.0, _rain(s["t"]), 0.0, 1800.0)
        s["t"] += 1.0
    _read(ctx, ctx.lib.frehg_re_get_field, (b"h", b"wc"), out)
    _read(ctx, ctx.lib.frehg_swe_get_field, (b"eta",), out[2:])
    got = {"h": out[0].inner, "wc": out[1].inner, "eta": out[2].inner}
    if c["solute"]:
        _read(ctx, ctx.lib.frehg_solute_get_field, (b"surface", b"subsurface"), out[3:])
        got.update(surface=out[3].inner, subsurface=out[4].inner)
    return got


def _batch(c, seed):
    """A batch of the network's inputs and targets and its weights (Glorot-uniform, small biases)."""
    rng = np.random.Generator(np.random.Philox(int(seed) % (1 << 40)))
    sd = np.array([1.0, .2, .2, .2, .2, .1, .1, 2.0, .05, .05, .01], dtype=np.float32)
    x = (rng.standard_normal((c["batch"], 11)).astype(np.float32) * sd - np.float32(0.5) * sd)
    y = (0.01 * np.tanh(x[:, 1] + x[:, 2] - x[:, 5]) + 0.002 * rng.standard_normal(c["batch"])).astype(np.float32)
    w = []
    for fan in ((64, 11), (64, 64), (1, 64)):
        lim = math.sqrt(6.0 / sum(fan))
        w += [rng.uniform(-lim, lim, fan).ravel(), rng.uniform(-0.1, 0.1, fan[0])]
    norm = np.concatenate([-0.5 * sd, [0.0], sd, [0.01]]).astype(np.float32)
    return x, y, np.concatenate(w).astype(np.float32), norm


def _prepare_mlp(c, seed):
    x, y, w, norm = _batch(c, seed)
    ctx = gpu.Context(0)
    ctx.mlp_init(1)
    ctx.mlp_set_params(w, norm)
    return {"run": _run_mlp, "ctx": ctx, "x": x, "y": y}


def _run_mlp(s):
    loss, grad = s["ctx"].mlp_loss_grad(s["x"], s["y"])
    return {"loss": loss, "grad": grad, "out": s["ctx"].mlp_predict(s["x"])}


# ---- what a pass cannot do without -----------------------------------------------------------------
def work(c):
    """Bytes: a solve reads its operator and right-hand side and writes its solution once; a time step reads and
    writes its state (heads and water contents; depth and velocities; concentrations) once and reads the
    conductivities or the bed once. Flops: the network's products."""
    k = c["kind"]
    if k == "solve":
        n = c["nx"] * c["ny"] * c["nz"]
        return {"bytes": 8.0 * n * (2 * c["ndim"] + 3), "flops": 0.0}
    if k == "mlp":
        return {"bytes": c["batch"] * 52.0, "flops": c["batch"] * 2.0 * 4 * (11 * 64 + 64 * 64 + 64)}
    if k == "ensemble":
        shape = np.random.Generator(np.random.Philox(3))
        n = 0
        for _ in range(c["boxes"]):
            nx, ny = shape.integers(c["lo"], c["hi"] + 1, size=2)
            n += int(nx) * int(ny) * int(shape.integers(20, 121))
        return {"bytes": 40.0 * n * c["steps"], "flops": 0.0}
    if k == "swe":
        return {"bytes": 56.0 * c["nx"] * c["ny"] * c["steps"], "flops": 0.0}
    n = c["nx"] * c["ny"] * c["nz"]
    if k == "re":
        return {"bytes": (32.0 + (8.0 if c["soil"] == "ks" else 0.0)) * n * c["steps"], "flops": 0.0}
    more = 16.0 if c["solute"] else 0.0
    return {"bytes": ((40.0 + more) * n + (56.0 + more) * c["nx"] * c["ny"]) * c["steps"], "flops": 0.0}


def tolerance(c):
    """Solves stop at a relative preconditioned residual of 1e-10 (groundwater) or 1e-12 (surface), and Picard
    loops at 1e-8 m: about four times what the mixed-precision solver and BiCGSTAB differ by from FP64 CG (the
    velocities of thin surface flow most). The network multiplies in BF16 (training) and FP16 (prediction)."""
    return {"solve": {"rel": 1e-9, "max": 1e-8},
            "re": {"rel": 2e-9, "max": 1e-7},
            "ensemble": {"rel": 1e-9, "max": 1.2e-7},
            "swe": {"rel": 4e-7, "max": 2e-6},
            "coupled": {"rel": 1e-9, "max": 1e-7},
            "mlp": {"rel": 1e-2, "max": 1e-1}}[c["kind"]]


# ---- the same in 64 bits, in plain torch ----------------------------------------------------------
def exact(c, seed):
    """Solves, groundwater runs and the network. The surface and coupled steps have none: their restatement
    (wetting and drying, limiters, drag, boundary rules) would be as long as the solver."""
    k = c["kind"]
    if k == "solve":
        op = _operator(c, seed)
        return _cg(op, op["b"])
    if k == "mlp":
        return _exact_mlp(c, seed)
    if k == "re":
        p, soils, idx, ks, h, wc = _re_setup(c, seed)
        if c["nx"] * c["ny"] * c["nz"] * c["steps"] > 2.0e7:
            return None
        h, wc, dt = _exact_re(p, soils, idx, ks, h, wc, c["steps"])
        return {"h": h, "wc": wc, "dt": dt}
    if k == "ensemble":
        out = []
        for nx, ny, nz, p, soil, ks, h0 in _boxes(c, seed):
            out.append(_exact_re(p, [soil], None, ks, np.full((nz, ny, nx), h0), None, c["steps"])[0])
        return out
    return None


def _exact_mlp(c, seed):
    x, y, w, norm = (torch.from_numpy(a).double() for a in _batch(c, seed))
    w.requires_grad_(True)
    W1, b1, W2, b2, w3, b3 = torch.split(w, [704, 64, 4096, 64, 64, 1])
    z = (x - norm[:11]) / norm[12:23]
    o = torch.tanh(torch.tanh(z @ W1.view(64, 11).T + b1) @ W2.view(64, 64).T + b2) @ w3 + b3
    loss = ((o - (y - norm[11]) / norm[23]) ** 2).mean()
    loss.backward()
    return {"loss": float(loss), "grad": w.grad, "out": (o * norm[23] + norm[11]).detach()}


class _Soil:
    """van Genuchten relations on (nz, ny, nx) fields."""

    def __init__(self, soils, idx, ks, shape):
        i = torch.zeros(shape, dtype=torch.long, device=DEV) if idx is None else \
            torch.from_numpy(np.asarray(idx)).long().to(DEV).reshape(shape)
        for name in ("alpha", "n", "theta_s", "theta_r", "Ss", "air_entry", "Ks_x", "Ks_y", "Ks_z"):
            setattr(self, name, torch.tensor([getattr(s, name) for s in soils], dtype=torch.float64, device=DEV)[i])
        if ks is not None:
            self.Ks_x = self.Ks_y = self.Ks_z = torch.from_numpy(np.asarray(ks)).to(DEV).reshape(shape)
        self.m = 1 - 1 / self.n

    def theta(self, h):
        se = (1 + (self.alpha * h).abs() ** self.n) ** -self.m
        return torch.where(h > self.air_entry, self.theta_s, self.theta_r + (self.theta_s - self.theta_r) * se)

    def kr(self, h):
        p = (self.alpha * h).abs() ** self.n
        t = -torch.expm1(self.m * torch.log(p / (1 + p)))
        return torch.where(h >= 0, torch.ones_like(h), (1 + p) ** (-self.m / 2) * t * t)

    def cap(self, h):
        a = (self.alpha * h).abs()
        c = self.alpha * self.n * self.m * (self.theta_s - self.theta_r) * a ** (self.n - 1) / (1 + a ** self.n) ** (self.m + 1)
        return torch.where(h > 0, torch.zeros_like(h), c)

    def head(self, w):
        th = torch.maximum(w, self.theta_r + 1e-7)
        x = (self.theta_s - self.theta_r) / (th - self.theta_r)
        h = -((x ** (1 / self.m) - 1).clamp_min(0) ** (1 / self.n)) / self.alpha
        return torch.where(th < self.theta_s, h, torch.zeros_like(h))

    def dkdw(self, w):
        th = torch.where((w > 0.9999 * self.theta_s) & (w < self.theta_s), 0.9999 * self.theta_s, w)
        se, m = (th - self.theta_r) / (self.theta_s - self.theta_r), self.m
        u = 1 - se ** (1 / m)
        t0 = u ** m
        t1 = 0.5 * self.Ks_z * se ** -0.5 * (1 - t0) ** 2
        t2 = 2 * self.Ks_z * se ** ((2 - m) / (2 * m)) * (1 - t0) * u ** (m - 1)
        return (t1 + t2) / (self.theta_s - self.theta_r)


def _mean(a, ax):
    lo, hi = [slice(None)] * 3, [slice(None)] * 3
    lo[ax], hi[ax] = slice(0, -1), slice(1, None)
    return 0.5 * (a[tuple(lo)] + a[tuple(hi)])


def _exact_re(p, soils, idx, ks, h, wc, steps):
    """The predictor-corrector (or Picard) groundwater step with lateral flow: closed sides, top head (1) or flux
    (2), closed (0) or free-drainage (3) bottom. Returns h, theta and the next dt."""
    shape = (h if h is not None else wc).shape
    S = _Soil(soils, idx, ks, shape)
    if h is not None:
        h = torch.from_numpy(h).to(DEV)
        w = S.theta(h)
    else:
        w = torch.from_numpy(wc).to(DEV)
        h = S.head(w)
    dx, dy, dz, bc4, bc5 = p.dx, p.dy, p.dz, p.bc_type[4], p.bc_type[5]
    V, Ax, Ay, Az, dt = dx * dy * dz, dy * dz, dx * dz, dx * dy, p.dt
    ss = S.Ss / S.theta_s
    first = True
    for _ in range(steps):
        hn, wn, hm = h, w, h
        for _ in range(p.picard_max):
            kr = S.kr(hm)
            kx, ky, kz = _mean(S.Ks_x * kr, 2), _mean(S.Ks_y * kr, 1), _mean(S.Ks_z * kr, 0)
            kbot = S.Ks_z[-1] * kr[-1] if bc4 else torch.zeros_like(kr[-1])
            ktop = S.Ks_z[0] if bc5 == 1 else S.Ks_z[0] * kr[0]
            st = S.cap(hm) + wn * ss
            D, b = st * V, st * hn * V
            off = []
            for K, ax, f in ((kx, 2, dt * Ax / dx), (ky, 1, dt * Ay / dy), (kz, 0, dt * Az / dz)):
                lo, hi = [slice(None)] * 3, [slice(None)] * 3
                lo[ax], hi[ax] = slice(0, -1), slice(1, None)
                m, q = torch.zeros_like(D), torch.zeros_like(D)
                m[tuple(hi)], q[tuple(lo)] = -f * K, -f * K
                D = D - m - q
                off.append((ax, m, q))
            gz = dt * V / dz
            b[:-1] -= kz * gz
            b[1:] += kz * gz
            b[-1] -= kbot * gz
            b[0] += ktop * gz
            if bc5 == 1:
                D[0] += ktop * dt * Az / (0.5 * dz)
                b[0] += ktop * dt * Az / (0.5 * dz) * p.htop
            else:
                b[0] -= (p.qtop + ktop) * gz
            hnew = _cg_3d(D, off, b, hm)
            d = float((hnew - hm).abs().max())
            hm = hnew
            if p.picard_max == 1 or d <= p.picard_tol:
                break
        hp, kr = hm, S.kr(hm)
        qx = Ax / dx * _mean(S.Ks_x * kr, 2) * (hp[:, :, 1:] - hp[:, :, :-1])
        qy = Ay / dy * _mean(S.Ks_y * kr, 1) * (hp[:, 1:] - hp[:, :-1])
        qz = torch.zeros((shape[0] + 1,) + tuple(shape[1:]), dtype=torch.float64, device=DEV)  # + = upward
        qz[1:-1] = Az * _mean(S.Ks_z * kr, 0) * ((hp[1:] - hp[:-1]) / dz - 1)
        qz[0] = p.qtop * Az if bc5 == 2 else Az * S.Ks_z[0] * ((hp[0] - p.htop) / (0.5 * dz) - 1)
        if bc4 == 3:
            qz[-1] = -Az * S.Ks_z[-1] * kr[-1]
        div = qz[1:] - qz[:-1]
        div[:, :, :-1] += qx
        div[:, :, 1:] -= qx
        div[:, :-1] += qy
        div[:, 1:] -= qy
        wcor = (wn * V + dt * div) / (V * (1 + (hp - hn) * ss))
        th = S.theta(hp)
        sat = wcor >= S.theta_s
        cand = ~sat & (th >= S.theta_s)
        ghost = torch.zeros_like(sat[-1]) if first else wn[-1] >= S.theta_s[-1]
        prev = sat
        while True:
            adj = torch.zeros_like(sat)
            adj[:-1] |= sat[1:]
            adj[-1] |= ghost
            adj[:, :, :-1] |= sat[:, :, 1:]
            adj[:, :-1] |= sat[:, 1:]
            adj[1:] |= prev[:-1]
            adj[:, :, 1:] |= prev[:, :, :-1]
            adj[:, 1:] |= prev[:, :-1]
            if bc5 == 1 and p.htop >= 0:
                adj[0] = True
            nxt = torch.where(cand, adj, sat)
            if bool((nxt == prev).all()):
                break
            prev = nxt
        w = torch.where(sat, S.theta_s, torch.where(adj, th, wcor))
        h = torch.where(~sat & ~adj & (wcor < 0.9999 * S.theta_s), S.head(wcor), hp)
        w = torch.minimum(torch.maximum(w, S.theta_r), S.theta_s)
        first = False
        if p.adaptive_dt:
            e = div / Az
            e = e[1:].abs()
            dq = float((e * dt / dz).max())
            lim = torch.where(w[1:] < S.theta_s[1:], p.co_max * dz / S.dkdw(w)[1:], torch.full_like(e, 1e8))
            dt = dt * (0.75 if dq > 0.02 else 1.25 if dq < 0.01 else 1.0)
            dt = max(min(dt, float(lim.min()), p.dt_max), p.dt_min)
    return h, w, float(dt)


def _cg_3d(D, off, b, x):
    def A(v):
        y = D * v
        for ax, m, q in off:
            lo, hi = [slice(None)] * 3, [slice(None)] * 3
            lo[ax], hi[ax] = slice(0, -1), slice(1, None)
            y[tuple(hi)] += m[tuple(hi)] * v[tuple(lo)]
            y[tuple(lo)] += q[tuple(lo)] * v[tuple(hi)]
        return y

    stop = 1e-14 * float((b / D).norm())
    r = b - A(x)
    z = r / D
    pv, rz = z.clone(), (r * z).sum()
    for _ in range(2000):
        if float(z.norm()) <= stop:
            break
        q = A(pv)
        a = rz / (pv * q).sum()
        x, r = x + a * pv, r - a * q
        z = r / D
        new = (r * z).sum()
        pv, rz = z + (new / rz) * pv, new
    return x
