"""The rarefaction integration of the exact Riemann solver against the oracle,
bit for bit, where its step control and its fast arithmetic change over:
weak to near-vacuum expansions (steps limited by the error, by the tenfold
growth, by the remaining pressure and by the smallest step), states outside
the range of the fast arithmetic, and solves that end in the non-adaptive
pass.  Every pair of SG and NASG materials, and a pair with a Mie-Grueneisen
one, which the fast arithmetic leaves out."""
import numpy as np
import pytest

import oracle_lib as ol
from m2c_amd import abi, configs

pytestmark = pytest.mark.gpu

SG, NASG = abi.material("SG", **configs.WATER_SG), abi.material("NASG", **configs.WATER_NASG)
AIR, HEAVY = abi.material("SG", **configs.AIR_SG), abi.material("SG", gamma=1.667)
MG = abi.material("MG", rho0=1000.0, c0=1500.0, s=1.6, Gamma0=0.9)
PAIRS = {"sg-air": (SG, AIR, 1000.0, 1.2, 1e5), "nasg-air": (NASG, AIR, 1000.0, 1.2, 1e5),
         "air-gas": (AIR, HEAVY, 1.0, 0.3, 1.0), "mg-air": (MG, AIR, 1000.0, 1.2, 1e5)}


def _problems(pair, n, seed, speed, scale=1.0):
    """Sides moving apart (or together) at `speed` times the slower sound speed."""
    a, b, ra, rb, p0 = PAIRS[pair]
    rng = np.random.default_rng(seed)
    Vm, Vp = np.zeros((n, 5)), np.zeros((n, 5))
    for V, r in ((Vm, ra), (Vp, rb)):
        V[:, 0] = scale * r * np.exp(rng.uniform(-0.3, 0.3, n))
        V[:, 4] = scale * p0 * 10 ** rng.uniform(-2, 2, n)
    c = np.sqrt(Vp[:, 4] / Vp[:, 0])
    Vp[:, 1] = rng.uniform(-0.2, 1.0, n) * speed * c
    Vm[:, 1] = -rng.uniform(-0.2, 1.0, n) * speed * c
    dirs = np.zeros((n, 3))
    dirs[:, 0] = 1.0
    return abi.materials(a, b), (dirs, Vm, np.zeros(n, dtype=np.int32), Vp, np.ones(n, dtype=np.int32))


def _check(mats, prob, **kw):
    from m2c_amd import runtime
    s = abi.default_scheme(**kw)
    g = runtime.Solver(abi.grid((4, 4, 4)), mats, 2, s).riemann_batch(*prob)
    o = ol.riemann_batch(mats, 2, s, *prob)
    ran = g["err"] != -2  # an integration path longer than the device's buffer
    assert np.mean(ran) > 0.5
    for key in ("Vs", "Vsm", "Vsp", "id", "err", "iters", "fevals"):
        x, y = g[key][ran], o[key][ran]
        bad = np.nonzero(~((x == y) | (np.isnan(x) & np.isnan(y))))[0]
        assert bad.size == 0, (key, bad[:5], x[bad[:3]], y[bad[:3]])


@pytest.mark.parametrize("pair", list(PAIRS))
@pytest.mark.parametrize("speed", [1e-6, 0.1, 1.0, 3.0])
@pytest.mark.parametrize("tol", [1e-5, 1e-10])
def test_expansions(pair, speed, tol):
    mats, prob = _problems(pair, 400, int(10 * speed) + 1, speed)
    _check(mats, prob, riem_tol_main=tol)


@pytest.mark.parametrize("steps,tol_rare", [(2, 1e-8), (20, 1e-3), (200, 1e-12), (1000, 1e-8)])
def test_integration_settings(steps, tol_rare):
    mats, prob = _problems("air-gas", 200, steps, 0.7)
    _check(mats, prob, riem_steps_rarefaction=steps, riem_tol_rarefaction=tol_rare)


@pytest.mark.parametrize("scale", [1e-60, 1e-30, 1e30, 1e60])
def test_states_outside_the_fast_range(scale):
    mats, prob = _problems("air-gas", 200, 3, 0.7, scale)
    _check(mats, prob, riem_min_pressure=-1e-8 * scale, riem_pressure_at_failure=1e-8 * scale)


@pytest.mark.parametrize("pair", ["sg-air", "nasg-air"])
@pytest.mark.parametrize("scale", [1e-60, 1e-30, 1e30, 1e60])
def test_liquid_states_outside_the_fast_range(pair, scale):
    """Gas pressures and densities far from the liquid's constants, the liquid
    itself near its density (NASG has a largest one)."""
    mats, (dirs, Vm, idm, Vp, idp) = _problems(pair, 200, 3, 0.7)
    Vp[:, 0] *= scale
    Vp[:, 4] *= scale
    _check(mats, (dirs, Vm, idm, Vp, idp), riem_min_pressure=-1e-8 * scale, riem_pressure_at_failure=1e-8 * scale)


def test_solves_that_end_in_the_second_pass():
    """Two iterations are too few: every problem is solved again without step
    control."""
    mats, prob = _problems("nasg-air", 200, 9, 0.5)
    _check(mats, prob, riem_maxits_main=2, riem_tol_main=1e-13)
