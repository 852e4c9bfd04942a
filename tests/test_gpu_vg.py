"""The device's van Genuchten relations (theta, C and K/Ks of a head, the head of a water content) against
50-digit values of their closed forms (src/re/VanGenuchten.hpp:18-137), from almost saturated to air-dry
soil, over the classes that the workloads use. The bounds are a few units in the last place: the relations are
evaluated with logarithms kept to more than double precision, so that neither powers with large exponents nor
1 - (p / (1 + p))^m in dry soil lose digits."""
import numpy as np
import pytest

from frehg_amd import abi, gpu

mp = pytest.importorskip("mpmath")
pytestmark = pytest.mark.gpu

CLASSES = [(2.0, 1.8), (0.5, 1.2), (3.35, 2.0), (5.0, 2.8), (1.43, 1.56)]
TS, TR = 0.40, 0.05


def exact(alpha, n, h):
    a = abs(mp.mpf(float(np.float64(alpha) * np.float64(h))))
    m = mp.mpf(1.0 - 1.0 / n)  # the class constant, rounded
    al, n = mp.mpf(alpha), mp.mpf(n)
    p = a ** n
    se = (1 + p) ** -m
    t = -mp.expm1(m * mp.log(p / (1 + p)))
    ts, tr = mp.mpf(TS), mp.mpf(TR)
    return tr + (ts - tr) * se, al * n * m * (ts - tr) * p * se / (a * (1 + p)), mp.sqrt(se) * t * t


@pytest.mark.parametrize("alpha,n", CLASSES)
def test_relations_against_50_digits(alpha, n):
    mp.mp.dps = 50
    nx = 400
    # below the air entry value (-0.02 m), above which theta is theta_s by the reference's rule
    h = -np.exp(np.linspace(np.log(0.021), np.log(1e6), nx))
    soil = abi.soil_params(alpha=alpha, n=n, theta_s=TS, theta_r=TR, Ks_x=1.0, Ks_y=1.0, Ks_z=1.0, Ss=0.0)
    ctx = gpu.Context(0)
    # one layer with a free-drainage bottom: its bottom face carries the cell's own K; dt = 1e-25 s keeps the head
    p = abi.re_params(soil=soil, solver=abi.solver_config(1e-13), bc_type=(0, 0, 0, 0, 3, 0), dz=1.0, dt=1e-25,
                      dt_min=1e-30, adaptive_dt=0, use_full3d=0)
    ctx.re_init(nx, 1, 1, p)
    ctx.re_set_initial(h=h)
    inner = lambda f: ctx.re_get(f).reshape(3, 3, nx + 2)[1, 1, 1:-1]
    wch, ch, wc, hwc = inner("wch"), inner("ch"), inner("wc"), inner("hwc")
    ctx.re_step()
    kz = inner("Kz")
    worst = [0.0] * 4
    for i in range(nx):
        th, c, kr = exact(alpha, n, h[i])
        # kr moves by up to 4 n relative units per unit of the solved head, which rounds by up to 2 ulps
        for q, (got, want, tol) in enumerate(((wch[i], th, 4e-16), (ch[i], c, 1.5e-15), (kz[i], kr, 2e-15 + 2e-15 * n))):
            err = abs(float((mp.mpf(float(got)) - want) / want))
            worst[q] = max(worst[q], err)
            assert err <= tol, (q, h[i], err)
        # the head of the stored water content, exact for the rounded quotient that the relation starts from
        w = float(wc[i])
        if w - TR >= 1e-7 and w < TS:
            x = mp.mpf((TS - TR) / (w - TR))
            m = 1 - 1 / mp.mpf(n)
            want = -((x ** (1 / m) - 1) ** (1 / mp.mpf(n))) / mp.mpf(alpha)
            # (1/m, 1/n and 1/alpha are rounded class constants: their exponents act on log x <= 15)
            err = abs(float((mp.mpf(float(hwc[i])) - want) / want))
            worst[3] = max(worst[3], err)
            assert err <= 2e-15 + 15 * 2.3e-16 / (1 - 1 / n) / n, (h[i], err)
    print(f"alpha {alpha} n {n}: theta {worst[0]:.1e} C {worst[1]:.1e} kr {worst[2]:.1e} head {worst[3]:.1e}")


def test_limits():
    """Zero and positive heads are saturated, theta_s gives head 0, and a NaN head stays NaN."""
    soil = abi.soil_params(alpha=2.0, n=1.8, theta_s=TS, theta_r=TR, Ks_z=1e-5)
    h = np.array([0.0, 1.0, -1e-300, -1e-18, -0.02, np.nan, -1e30])
    ctx = gpu.Context(0)
    ctx.re_init(len(h), 1, 1, abi.re_params(soil=soil, adaptive_dt=0))
    ctx.re_set_initial(h=h)
    inner = lambda f: ctx.re_get(f).reshape(3, 3, len(h) + 2)[1, 1, 1:-1]
    wch, ch, hwc = inner("wch"), inner("ch"), inner("hwc")
    assert (wch[:4] == TS).all() and (ch[:2] == 0.0).all() and (hwc[:4] == 0.0).all()
    assert np.isfinite(ch[2:5]).all() and np.isnan(wch[5]) and np.isnan(ch[5])
    assert wch[6] == pytest.approx(TR, rel=1e-12) and np.isfinite(ch[6])


@pytest.mark.parametrize("alpha,n", CLASSES)
def test_heads_whose_power_overflows(alpha, n):
    """(alpha |h|)^n beyond the largest double, just below it (where twice of it overflows), and an infinite head:
    theta is theta_r, as the closed form's limit."""
    edge = np.exp(np.log(1.797e308) / n) / alpha  # (alpha |h|)^n = 1.797e308
    h = -np.array([0.4 ** (1 / n) * edge, 0.7 ** (1 / n) * edge, 1.01 * edge, min(1e10 * edge, 1e300), np.inf])
    soil = abi.soil_params(alpha=alpha, n=n, theta_s=TS, theta_r=TR, Ks_z=1e-5)
    ctx = gpu.Context(0)
    ctx.re_init(len(h), 1, 1, abi.re_params(soil=soil, adaptive_dt=0))
    ctx.re_set_initial(h=h)
    wch = ctx.re_get("wch").reshape(3, 3, len(h) + 2)[1, 1, 1:-1]
    assert (wch == TR).all(), wch
