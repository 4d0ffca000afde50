"""The stage on tiles of one material and on mixed tiles, against the oracle,
bit for bit: every flux, limiter, equation of state and boundary condition on
grids that tiles do not divide, thinner than a tile and its halo, with
inactive cells in a one-material solver, with states at the ends of the fast
arithmetic's range, and shock-bubbles whose grids hold both kinds of tile."""
import numpy as np
import pytest

import oracle_lib as ol
from m2c_amd import abi, configs

pytestmark = pytest.mark.gpu

MATS = {
    "sg": abi.material("SG", gamma=1.4),
    "stiff": abi.material("SG", gamma=6.12, pc=3.43, pmin=-3.0),
    "nasg": abi.material("NASG", gamma=1.19, pc=6.2, b=0.05, q=-1.2),
    "mg": abi.material("MG", rho0=1.0, c0=2.0, s=1.3, Gamma0=1.2),
}
BCS = (abi.BC_INLET, abi.BC_OUTLET, abi.BC_SYMMETRY, abi.BC_SLIPWALL, abi.BC_STICKWALL, abi.BC_INLET2)


def _inner(a):
    return a[1:-1, 1:-1, 1:-1]


def _state(n, seed, rough):
    rng = np.random.default_rng(seed)
    V = np.zeros((n[2] + 2, n[1] + 2, n[0] + 2, 5))
    amp = 0.3 if rough else 0.02
    V[..., 0] = 1.1 * np.exp(rng.uniform(-amp, amp, V.shape[:3]))
    V[..., 1:4] = rng.uniform(-amp, amp, V.shape[:3] + (3,)) + (2.5 if rough else 0.0) * np.array([1.0, -1.0, 0.5])
    V[..., 4] = np.exp(rng.uniform(-amp, amp, V.shape[:3]))
    return V


def _pair(n, mat, V, ID=None, nmat=1, **kw):
    from m2c_amd import runtime
    g = abi.grid(n, (0, 0, 0), tuple(0.1 * a for a in n), BCS, inlet=[1.0, 0.2, 0.1, -0.1, 1.2],
                 inlet2=[1.2, -0.1, 0.3, 0.2, 0.9])
    mats = abi.materials(mat)
    s = abi.default_scheme(**kw)
    if ID is None:
        ID = np.zeros(V.shape[:3], dtype=np.int32)
    configs.fill_ghosts(V, ID, None, g)
    o = ol.Oracle(g, mats, nmat, s)
    o.set_state(V, ID, None)
    gpu = runtime.Solver(g, mats, nmat, s)
    gpu.set_state(V, ID, None)
    return gpu, o


def _same_residual(gpu, o):
    try:
        Ro = _inner(o.residual())
    except RuntimeError as e:
        from m2c_amd import runtime
        assert "hyperbolicity" in str(e)
        with pytest.raises(runtime.M2CError, match="error -4"):
            gpu.compute_residual()
        return
    Rg = _inner(gpu.compute_residual())
    assert np.array_equal(Rg, Ro, equal_nan=True), np.nanmax(np.abs(Rg - Ro))


@pytest.mark.parametrize("mat", list(MATS))
@pytest.mark.parametrize("flux", [abi.FLUX_HLLC, abi.FLUX_ROE, abi.FLUX_LLF])
@pytest.mark.parametrize("limiter", [abi.LIM_VANALBADA, abi.LIM_GMM, abi.LIM_NONE])
@pytest.mark.parametrize("rough", [False, True])
def test_one_material(mat, flux, limiter, rough):
    n = (35, 11, 9)
    gpu, o = _pair(n, MATS[mat], _state(n, 5, rough), flux=flux, limiter=limiter)
    for v in range(4):
        gpu.set_tile(v)
        _same_residual(gpu, o)


VARS = [abi.VAR_CONSERVATIVE, abi.VAR_PRIMITIVE_CHARACTERISTIC, abi.VAR_CONSERVATIVE_CHARACTERISTIC]


@pytest.mark.parametrize("mat", list(MATS))
@pytest.mark.parametrize("var", VARS)
@pytest.mark.parametrize("flux,limiter", [(abi.FLUX_HLLC, abi.LIM_VANALBADA), (abi.FLUX_ROE, abi.LIM_GMM),
                                          (abi.FLUX_LLF, abi.LIM_NONE)])
@pytest.mark.parametrize("rough", [False, True])
def test_reconstruction_variables(mat, var, flux, limiter, rough):
    """Rough states send some cells back to primitive variables, also cells
    around a tile whose faces the tile forms."""
    for n in ((35, 11, 9), (5, 3, 2)):
        gpu, o = _pair(n, MATS[mat], _state(n, 6, rough), flux=flux, limiter=limiter, var_type=var)
        _same_residual(gpu, o)


@pytest.mark.parametrize("var", VARS)
@pytest.mark.parametrize("overlap", [True, False])
def test_reconstruction_variables_with_an_interface(var, overlap):
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, Phi = configs.c2_shock_bubble(32, radius=0.27)
    s.var_type, s.flux, s.limiter = var, abi.FLUX_ROE, abi.LIM_GMM
    o = ol.Oracle(g, mats, nmat, s)
    o.set_state(V, ID, Phi)
    gpu = runtime.Solver(g, mats, nmat, s)
    gpu.set_overlap(overlap)
    gpu.set_state(V, ID, Phi)
    gpu.run_steps(3)
    o.run_steps(3)
    for a, b in zip(gpu.get_state(), o.get_state()):
        assert np.array_equal(_inner(a), _inner(b))


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (1, 3, 1), (1, 1, 5), (33, 1, 1), (8, 8, 4), (9, 9, 5), (7, 65, 3)])
@pytest.mark.parametrize("ti", [abi.TI_FE, abi.TI_RK2, abi.TI_RK3])
def test_small_and_ragged_grids(n, ti):
    gpu, o = _pair(n, MATS["stiff"], _state(n, 8, False), integrator=ti, time_step=2e-3)
    for v in range(4):
        gpu.set_tile(v)
        gpu.run_steps(1)
        o.run_steps(1)
        assert np.array_equal(_inner(gpu.get_state()[0]), _inner(o.get_state()[0])), v


def test_inactive_cells_in_a_one_material_solver():
    """Material number nmat marks inactive cells; a solver of one material
    learns of them when the IDs are uploaded, also between steps."""
    n = (40, 18, 13)
    V = _state(n, 3, False)
    gpu, o = _pair(n, MATS["sg"], V, integrator=abi.TI_RK2, cfl=0.3)
    gpu.run_steps(1)
    o.run_steps(1)
    assert np.array_equal(_inner(gpu.get_state()[0]), _inner(o.get_state()[0]))
    ID = np.zeros(V.shape[:3], dtype=np.int32)
    ID[5:8, 7:9, 20:23] = 1
    ID[:, 3, 3] = 1
    gpu.upload(abi.FIELD_ID, ID)
    o.set_state(o.get_state()[0], ID, None)
    live = _inner(ID) == 0
    for v in range(4):
        gpu.set_tile(v)
        _g, _o = _inner(gpu.compute_residual()), _inner(o.residual())
        assert np.array_equal(_g[live], _o[live]), v


def test_solvers_of_one_table_on_every_kernel():
    """Solvers of the same materials, which no other test has, one after another
    on each form of the stage, all alive: each form finds the table."""
    n = (20, 12, 9)
    V = _state(n, 12, False)
    mat = abi.material("SG", gamma=1.37, pc=0.25)
    forms = [dict(), dict(flux=abi.FLUX_ROE), dict(var_type=abi.VAR_CONSERVATIVE_CHARACTERISTIC),
             dict(rec_type=abi.REC_CONSTANT), dict(flux=abi.FLUX_GODUNOV)]
    pairs = []
    for kw in forms:
        pairs.append(_pair(n, mat, V, **kw))
        for gpu, o in pairs:
            _same_residual(gpu, o)
    ID = np.zeros(V.shape[:3], dtype=np.int32)
    ID[3:5, 4:6, 8:11] = 1
    for gpu, o in pairs:
        gpu.upload(abi.FIELD_ID, ID)
        o.set_state(V, ID, None)
        live = _inner(ID) == 0
        assert np.array_equal(_inner(gpu.compute_residual())[live], _inner(o.residual())[live])


@pytest.mark.parametrize("var", VARS)
def test_inactive_cells_in_other_variables(var):
    n = (40, 18, 13)
    V = _state(n, 8, True)
    gpu, o = _pair(n, MATS["stiff"], V, var_type=var)
    ID = np.zeros(V.shape[:3], dtype=np.int32)
    ID[5:8, 7:9, 20:23] = 1
    gpu.upload(abi.FIELD_ID, ID)
    o.set_state(V, ID, None)
    live = _inner(ID) == 0
    assert np.array_equal(_inner(gpu.compute_residual())[live], _inner(o.residual())[live])


@pytest.mark.parametrize("case", ["denormal", "tiny", "huge", "vacuum", "zeros"])
def test_ends_of_the_fast_range(case):
    """Velocities down to denormals (a wave's exponential front), states far
    outside the range that the fast arithmetic takes, and exact zeros."""
    n = (24, 10, 8)
    rng = np.random.default_rng(2)
    V = _state(n, 4, False)
    mag = rng.uniform(-1, 1, V.shape[:3] + (3,))
    if case == "denormal":
        V[..., 1:4] = mag * 10.0 ** rng.uniform(-323, -280, mag.shape)
    elif case == "tiny":
        V[..., 1:4] = mag * 10.0 ** rng.uniform(-300, -100, mag.shape)
        V[..., 4] *= 10.0 ** rng.uniform(-200, 0, V.shape[:3])
    elif case == "huge":
        V[..., 0] *= 1e60
        V[..., 4] *= 1e90
        V[..., 1:4] *= 1e15
    elif case == "vacuum":
        thin = 10.0 ** rng.uniform(-40, 0, V.shape[:3])
        V[..., 0] *= thin
        V[..., 4] *= thin
    else:
        V[..., 1:4] = 0.0
        V[:, :, 12:, 0], V[:, :, :12, 0] = 1.0, 0.5
        V[..., 4] = 1.0
    gpu, o = _pair(n, MATS["sg"], V)
    _same_residual(gpu, o)


# exponent ranges of density, velocities and pressure at the ends of the fast
# arithmetic, as factors on the state
RANGES = {"denormal": (0, (-323, -280), 0), "tiny": (0, (-300, -100), (-200, 0)), "huge": (60, 15, 90),
          "vacuum": ((-40, 0), 0, (-40, 0)), "thin": ((-40, 0), (-40, 0), 0), "hot": (0, 0, (0, 70))}


# NASG and MG have a largest density
@pytest.mark.parametrize("case,mat", [(c, m) for c in RANGES for m in MATS if c != "huge" or m in ("sg", "stiff")])
@pytest.mark.parametrize("flux,limiter,var", [
    (abi.FLUX_HLLC, abi.LIM_VANALBADA, abi.VAR_PRIMITIVE), (abi.FLUX_HLLC, abi.LIM_GMM, abi.VAR_PRIMITIVE),
    (abi.FLUX_ROE, abi.LIM_VANALBADA, abi.VAR_PRIMITIVE), (abi.FLUX_HLLC, abi.LIM_VANALBADA, abi.VAR_CONSERVATIVE),
    (abi.FLUX_HLLC, abi.LIM_VANALBADA, abi.VAR_PRIMITIVE_CHARACTERISTIC),
    (abi.FLUX_ROE, abi.LIM_GMM, abi.VAR_CONSERVATIVE_CHARACTERISTIC)])
def test_ends_of_the_fast_range_in_every_form(case, mat, flux, limiter, var):
    n = (24, 10, 8)
    rng = np.random.default_rng(11)
    V = _state(n, 4, False)
    for q, (r, c) in enumerate(zip(RANGES[case], (slice(0, 1), slice(1, 4), slice(4, 5)))):
        shape = V[..., c].shape
        if isinstance(r, tuple):
            V[..., c] = rng.uniform(0.1, 1.0, shape) * 10.0 ** rng.uniform(r[0], r[1], shape) * (1 if q != 1 else
                                                                                                 rng.choice([-1, 1], shape))
        elif r:
            V[..., c] *= 10.0 ** r
    gpu, o = _pair(n, MATS[mat], V, flux=flux, limiter=limiter, var_type=var)
    _same_residual(gpu, o)


@pytest.mark.parametrize("comp", [0, 1, 3, 4])
@pytest.mark.parametrize("mat", ["sg", "nasg"])
@pytest.mark.parametrize("value,flux,var", [
    (x, f, q) for f, q, xs in ((abi.FLUX_HLLC, abi.VAR_PRIMITIVE, (np.inf, -np.inf, np.nan)),
                               (abi.FLUX_HLLC, abi.VAR_CONSERVATIVE_CHARACTERISTIC, (np.inf, -np.inf, np.nan)),
                               (abi.FLUX_ROE, abi.VAR_PRIMITIVE, (np.nan,)), (abi.FLUX_LLF, abi.VAR_PRIMITIVE, (np.nan,)))
    for x in xs])
def test_infinities_and_nan(value, comp, mat, flux, var):
    """One such value in a cell: the same residual or the same abort.  (Roe and
    LLF in primitive variables with NaN alone: the reference aborts on an
    infinite density or pressure that clipping would replace, where these
    fluxes here go on.)"""
    n = (24, 10, 8)
    V = _state(n, 4, False)
    V[4, 5, 9, comp] = value
    gpu, o = _pair(n, MATS[mat], V, flux=flux, var_type=var)
    _same_residual(gpu, o)


@pytest.mark.parametrize("water", ["sg", "nasg"])
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_mixed_and_one_material_tiles(water, variant):
    """40^3 shock-bubble: tiles inside the gas, tiles of water and mixed ones,
    with the stage overlapped with the Riemann solve and after it."""
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, Phi = configs.c2_shock_bubble(40, radius=0.27)
    if water == "nasg":
        mats[0] = abi.material("NASG", **configs.WATER_NASG)
        r2, u2, p2 = configs.nasg_post_shock(1000.0, 1e5, *(configs.WATER_NASG[k] for k in ("gamma", "pc", "b", "q")),
                                             1.5)
        V[V[..., 1] > 0] = [r2, u2, 0.0, 0.0, p2]
    o = ol.Oracle(g, mats, nmat, s)
    o.set_state(V, ID, Phi)
    o.run_steps(3)
    Vo, IDo, Po = o.get_state()
    for overlap in (True, False):
        gpu = runtime.Solver(g, mats, nmat, s)
        gpu.set_overlap(overlap)
        gpu.set_tile(variant)
        gpu.set_state(V, ID, Phi)
        gpu.run_steps(3)
        Vg, IDg, Pg = gpu.get_state()
        assert np.array_equal(_inner(IDg), _inner(IDo)) and np.array_equal(_inner(Pg), _inner(Po))
        assert np.array_equal(_inner(Vg), _inner(Vo)), np.abs(_inner(Vg) - _inner(Vo)).max()


@pytest.mark.parametrize("integrator", [abi.TI_RK2, abi.TI_RK3])
@pytest.mark.parametrize("bandwidth", [None, 8])
def test_level_set_beside_the_riemann_launch(integrator, bandwidth):
    """Grids of 2^20 cells and more: the level set on the second stream, against
    the run on one stream."""
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, Phi = configs.c2_shock_bubble(102)
    s.integrator = integrator
    if bandwidth:
        s.ls_bandwidth = bandwidth
        s.reinit_frequency = 1
    out = []
    for overlap in (True, False):
        gpu = runtime.Solver(g, mats, nmat, s)
        gpu.set_overlap(overlap)
        gpu.set_state(V, ID, Phi)
        if bandwidth:
            gpu.construct_narrow_band()
        gpu.run_steps(2)
        out.append([np.array(a) for a in gpu.get_state()])
    for a, b in zip(*out):
        assert np.array_equal(_inner(a), _inner(b))
