"""Near-zero shocks in the exact Riemann solver: problems whose Hugoniot
bracket comes to rest at the spacing of doubles before the stopping rule is
met (quasi-static water / gas faces), where the device leaves the root
iteration at once and the oracle spends its whole budget.  Bit for bit the
oracle's states, iteration and evaluation counts, with budgets that end the
iteration before, at and after the point of rest."""
import numpy as np
import pytest

import oracle_lib as ol
from m2c_amd import abi, configs

pytestmark = pytest.mark.gpu


def _problems(n, seed, rho_water):
    rng = np.random.default_rng(seed)
    Vm, Vp = np.zeros((n, 5)), np.zeros((n, 5))
    Vm[:, 0], Vp[:, 0] = rho_water * np.exp(rng.uniform(-1e-3, 1e-3, n)), 1.2 * np.exp(rng.uniform(-0.1, 0.1, n))
    p = 1e5 * np.exp(rng.uniform(-0.5, 0.5, n))
    # jumps from one unit in the last place to a few per mille, velocities to match
    Vm[:, 4] = p
    Vp[:, 4] = p * (1.0 + 10 ** rng.uniform(-16, -2.5, n) * rng.choice([-1, 0, 1], n))
    Vm[:, 1] = 10 ** rng.uniform(-14, 0, n) * rng.choice([-1, 0, 1], n)
    Vp[:, 1] = 10 ** rng.uniform(-14, 0, n) * rng.choice([-1, 0, 1], n)
    dirs = np.zeros((n, 3))
    dirs[:, 0] = 1.0
    idm, idp = np.zeros(n, dtype=np.int32), np.ones(n, dtype=np.int32)
    flip = rng.random(n) < 0.5
    Vm[flip], Vp[flip] = Vp[flip].copy(), Vm[flip].copy()
    idm[flip], idp[flip] = 1, 0
    return dirs, Vm, idm, Vp, idp


@pytest.mark.parametrize("water", ["sg", "nasg"])
@pytest.mark.parametrize("budget", [1, 2, 3, 7, 20, 200])
def test_near_zero_shocks_bitwise(water, budget):
    from m2c_amd import runtime
    w = abi.material("SG", **configs.WATER_SG) if water == "sg" else abi.material("NASG", **configs.WATER_NASG)
    mats = abi.materials(w, abi.material("SG", **configs.AIR_SG))
    s = abi.default_scheme(riem_tol_main=1e-10, riem_maxits_shock=budget)
    prob = _problems(600, budget, 1000.0)
    g = runtime.Solver(abi.grid((4, 4, 4)), mats, 2, s).riemann_batch(*prob)
    o = ol.riemann_batch(mats, 2, s, *prob)
    # a solve that ends too early leaves the secant wandering, and its rarefaction
    # path can outgrow the device's buffer: reported as err = -2, no states
    ran = g["err"] != -2
    assert np.mean(ran) > 0.9
    for key in ("Vs", "Vsm", "Vsp", "id", "err", "iters", "fevals"):
        a, b = g[key][ran], o[key][ran]
        bad = np.nonzero(~((a == b) | (np.isnan(a) & np.isnan(b))))[0]
        assert bad.size == 0, (key, bad[:5], a[bad[:3]], b[bad[:3]])
    if budget == 200:
        assert np.sum(o["iters"] >= 200) > 5  # the secant stalls on some of them
