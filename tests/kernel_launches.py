"""Counts the kernels that steps of small solvers launch and the runtime calls
they make, by name, and prints them as JSON: {case: {name: calls}}.  Run as a program of its own: the
profiler belongs to torch, which has to bring up the runtime before the
library does."""
import json
import os
import re
import sys

import torch
from torch.profiler import ProfilerActivity, profile

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from m2c_amd import abi, configs, runtime  # noqa: E402


def counted(work):
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        work()
        torch.cuda.synchronize()
    out = {}
    for e in p.key_averages():
        m = re.search(r"m2c::(k_\w+)", e.key) or re.match(r"(hip\w+)$", e.key)
        if m:
            out[m.group(1)] = out.get(m.group(1), 0) + e.count
    return out


def bubble(overlap, **scheme):
    g, mats, nmat, s, V, ID, Phi = configs.c2_shock_bubble(24, radius=0.27)
    for k, v in scheme.items():
        setattr(s, k, v)
    sol = runtime.Solver(g, mats, nmat, s)
    sol.set_overlap(overlap)
    sol.set_state(V, ID, Phi)
    sol.run_steps(1)
    return counted(lambda: sol.run_steps(1))


def gas(inactive, **scheme):
    g, mats, nmat, s, V, ID, _ = configs.c1_sod((32, 8, 8))
    for k, v in scheme.items():
        setattr(s, k, v)
    sol = runtime.Solver(g, mats, nmat, s)
    ID = ID.copy()
    if inactive:
        ID[3:5, 3:5, 10:14] = nmat
    sol.set_state(V, ID)
    sol.run_steps(1)
    return counted(lambda: sol.run_steps(1))


def new_materials():
    """A solver with materials that no other has, then one of another flux."""
    g, _, _, s, _, _, _ = configs.c1_sod((16, 8, 8))
    mats = abi.materials(abi.material("SG", gamma=1.23))
    made = []
    first = counted(lambda: made.append(runtime.Solver(g, mats, 1, s)))
    s.flux = abi.FLUX_ROE
    return first, counted(lambda: made.append(runtime.Solver(g, mats, 1, s)))


def gas_again(way):
    """A solver of one gas that held inactive cells before."""
    g, mats, nmat, s, V, ID, _ = configs.c1_sod((32, 8, 8))
    sol = runtime.Solver(g, mats, nmat, s)
    state = (1.0, 0.0, 0.0, 0.0, 1.0)
    solid = abi.geometry("sphere", (0.4, 0.1, 0.1), radius=0.1, materialid=nmat, state=state)
    if way == "upload":
        held = ID.copy()
        held[3:5, 3:5, 10:14] = nmat
        sol.set_state(V, held)
    else:
        sol.initialize(state, 0, [solid])
    with_cells = counted(lambda: sol.run_steps(1))
    if way == "upload":
        sol.set_state(V, ID)
    else:
        sol.initialize(state, 0, [])
    return {"with": with_cells, "without": counted(lambda: sol.run_steps(1))}


def tuned(n, first, second):
    """The first step of a solver after another of its size tuned its tiles."""
    sols = []
    for scheme in (first, second):
        g, mats, nmat, s, V, ID, _ = configs.c1_sod(n)
        for k, v in scheme.items():
            setattr(s, k, v)
        sols.append(runtime.Solver(g, mats, nmat, s))
        sols[-1].set_state(V, ID)
    sols[0].autotune()
    return counted(lambda: sols[1].run_steps(1))


def main():
    torch.zeros(1, device="cuda")
    constant = dict(rec_type=abi.REC_CONSTANT)
    first, second = new_materials()
    out = {
        "bubble": bubble(True),
        "bubble, one stream": bubble(False),
        "bubble, constant": bubble(True, **constant),
        "bubble, constant, one stream": bubble(False, **constant),
        "gas": gas(False),
        "gas, inactive cells": gas(True),
        "gas, inactive cells, constant": gas(True, **constant),
        "new materials": first,
        "new materials, roe as well": second,
        "gas again, upload": gas_again("upload"),
        "gas again, initialize": gas_again("initialize"),
        "tuned by its like": tuned((64, 64, 65), {}, {}),
        "tuned by constant": tuned((64, 64, 66), constant, {}),
        "tuned by characteristic": tuned((64, 64, 67), dict(var_type=abi.VAR_CONSERVATIVE_CHARACTERISTIC), {}),
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
