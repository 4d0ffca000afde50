"""Fields to the device and back bit for bit, at sizes around the ones where
the copies change: below and above the threshold of the pinned ring, whole and
partial last chunks, fewer and more chunks than the ring holds, two solvers
copying from two threads at once, and a state stepped after an upload."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle_lib as ol
from m2c_amd import abi, configs

pytestmark = pytest.mark.gpu

# cells with ghosts x 40 B: 8 MB threshold, 2 MB chunks, a ring of 8
GRIDS = [(3, 2, 1), (57, 58, 58), (58, 58, 58), (102, 94, 98), (126, 126, 126), (158, 126, 126)]


def _fields(shape, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(shape + (5,)), rng.integers(0, 2, shape).astype(np.int32), rng.standard_normal(shape))


def _solver(n):
    from m2c_amd import runtime
    mats = abi.materials(abi.material("SG", gamma=1.4), abi.material("SG", gamma=1.667))
    return runtime.Solver(abi.grid(n), mats, 2, abi.default_scheme(n_levelsets=1))


@pytest.mark.parametrize("n", GRIDS)
def test_round_trip(n):
    sol = _solver(n)
    for seed in (1, 2):  # the second pass uses the ring again
        V, ID, Phi = _fields(sol.shape, seed)
        sol.set_state(V, ID, Phi)
        sol.upload(abi.FIELD_V1, V[::-1])
        Vd, IDd, Pd = sol.get_state()
        assert np.array_equal(Vd, V) and np.array_equal(IDd, ID) and np.array_equal(Pd, Phi)
        assert np.array_equal(sol.download(abi.FIELD_V1), V[::-1])
        sol.upload_levelset(0, Phi[::-1])
        assert np.array_equal(sol.download_levelset(0), Phi[::-1])


def test_two_solvers_from_two_threads():
    sols = [_solver((126, 126, 126)) for _ in range(2)]
    bad = []

    def work(q):
        for seed in range(3):
            V, ID, Phi = _fields(sols[q].shape, 10 * q + seed)
            sols[q].set_state(V, ID, Phi)
            out = sols[q].get_state()
            if not all(np.array_equal(a, b) for a, b in zip(out, (V, ID, Phi))):
                bad.append((q, seed))

    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_steps_between_large_copies():
    from m2c_amd import runtime
    g, mats, nmat, s, V, ID, _ = configs.c1_sod((96, 64, 64))
    gpu = runtime.Solver(g, mats, nmat, s)
    gpu.set_state(V, ID)
    gpu.run_steps(2)
    o = ol.Oracle(g, mats, nmat, s)
    o.set_state(V, ID, None)
    o.run_steps(2)
    assert np.array_equal(gpu.get_state()[0][1:-1, 1:-1, 1:-1], o.get_state()[0][1:-1, 1:-1, 1:-1])


@pytest.mark.parametrize("n", [(58, 58, 58), (126, 126, 126)])
def test_pinned_arrays_of_the_caller(n):
    """Fields to and from arrays the caller has pinned (through the runtime
    that the library has loaded, see test_zz_no_alloc.py)."""
    sol = _solver(n)
    hip = C.CDLL("libamdhip64.so.7")
    V, ID, Phi = _fields(sol.shape, 3)
    same = []
    for field, a in ((abi.FIELD_V, V), (abi.FIELD_ID, ID), (abi.FIELD_PHI, Phi)):
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(a.nbytes), 0) == 0
        C.memmove(p, a.ctypes.data, a.nbytes)
        sol._check(sol.L.m2cx_upload(sol.h, field, p))
        C.memset(p, 0xFF, a.nbytes)
        sol._check(sol.L.m2cx_download(sol.h, field, p))
        same.append(C.string_at(p, a.nbytes) == a.tobytes())
        assert hip.hipHostFree(p) == 0
    assert same == [True, True, True]
