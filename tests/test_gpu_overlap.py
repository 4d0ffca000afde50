"""The level set beside the Riemann launch where the launch reads it: level-set
and average normals, on grids of 2^20 cells and more (from where the last
stage's level set runs on the second stream), against the run on one stream.
The Riemann launch gets 256 lanes, each with many faces one after another, so
that it still takes normals from the level set long after the stage's tiles of
one material are done."""
import numpy as np
import pytest

import levelset_cases as lc
from m2c_amd import abi, configs

pytestmark = pytest.mark.gpu


def _inner(a):
    return a[1:-1, 1:-1, 1:-1]


def _same_on_one_stream(monkeypatch, build, steps=2):
    out = []
    for overlap in (False, True):
        if overlap:
            monkeypatch.setenv("M2C_RIEMANN_LANES", "256")
        sol, levels = build()
        sol.set_overlap(overlap)
        sol.run_steps(steps)
        out.append([np.array(a) for a in sol.get_state()] + [sol.download_levelset(q) for q in range(1, levels)])
        assert sol.counters()["riemann_calls"] > 256 * 3 * steps
        sol.close()
    for a, b in zip(*out):
        assert np.array_equal(_inner(a), _inner(b))


@pytest.mark.parametrize("normal", [abi.RNORMAL_LEVEL_SET, abi.RNORMAL_AVERAGE])
@pytest.mark.parametrize("integrator", [abi.TI_RK2, abi.TI_RK3])
@pytest.mark.parametrize("solver", [abi.LSSOLVER_FINITE_DIFFERENCE, abi.LSSOLVER_FINITE_VOLUME])
def test_normals_from_the_level_set(monkeypatch, normal, integrator, solver):
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, Phi = configs.c2_shock_bubble(102, radius=0.1)
    # a moving bubble with a tangential slip: the interface problems depend on
    # the direction from the first step
    V[..., 1] += 30.0
    V[..., 2] -= 20.0
    V[ID == 1, 3] += 15.0
    s.riemann_normal, s.integrator, s.ls_solver = normal, integrator, solver

    def build():
        sol = runtime.Solver(g, mats, nmat, s)
        sol.set_state(V, ID, Phi)
        return sol, 1

    _same_on_one_stream(monkeypatch, build)


def test_normals_from_two_level_sets(monkeypatch):
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, phis, ls, _ = lc.two_bubbles(
        n=(164, 81, 80), mat2=abi.material("SG", gamma=1.667), rnormal=abi.RNORMAL_LEVEL_SET, radii=(0.12, 0.1),
        shocks=(0.35, 1.7))
    V[..., 2] -= 20.0
    V[ID > 0, 3] += 15.0
    configs.fill_ghosts(V, ID, None, g)

    def build():
        sol = runtime.Solver(g, mats, nmat, s, levelsets=ls)
        sol.set_state(V, ID, phis[0])
        sol.upload_levelset(1, phis[1])
        return sol, 2

    _same_on_one_stream(monkeypatch, build)
