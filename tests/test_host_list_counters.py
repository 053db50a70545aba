"""The counters of the deferred lists (faces of each sweep, and the two of the
cells that the u2p passes of a step alternate between) are each cleared before
their first use of a step: with every buffer poisoned, the host executor's steps
stop at a stale counter, and otherwise give the oracle's state."""
import os
import subprocess

import numpy as np
import pytest

import host_grid as H
from koral_amd import params as KP, problems as PR, grid as GR


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("hp") / "grid_check_poison"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fopenmp", "-ffp-contract=off", "-fno-fast-math", "-I",
                    os.path.join(H.ROOT, "koral_amd", "csrc"), "-I", os.path.join(H.ROOT, "include"),
                    os.path.join(H.ROOT, "tests", "host", "grid_check_poison.cpp"), "-o", str(out)], check=True)
    return str(out)


# a tube of fewer than four cells takes the launches that clear on their own
@pytest.mark.parametrize("kind,tune", [("tube", None), ("tube3", None), ("torus", None), ("tube", "combrt"),
                                       ("torus", "combrt")])
def test_counters_cleared_before_use(oracle, exe, tmp_path, kind, tune):
    if kind == "torus":
        P = KP.params_torus_mhd()
        spec, p = PR.torus_setup(P, n=(12, 10, 4))
    else:
        P = KP.params_tube()
        spec, p = PR.tube_setup(P, nx=3 if kind == "tube3" else 24)
    p = GR.to_aos(p)
    S = oracle.GridState(P, oracle.Grid(spec), p)
    S.init_u()
    S.set_bc()
    dt = 1. / S.tstepden()
    t = 0.
    for _ in range(2):
        tm, _ = S.step(t, dt)
        t += dt
        dt = 1. / tm
    inp, out = tmp_path / "in.bin", tmp_path / "out.bin"
    H.write_input(inp, P, spec, p)
    r = H.run(exe, inp, out, 0, 1, "step", 2, timeout=600, tune=tune)
    assert r.returncode == 0, r.stderr[-3000:]
    pd, ud, fd, _ = H.read_output(out, spec, P.nv, 2)
    assert np.array_equal(pd, S.p, equal_nan=True) and np.array_equal(ud, S.u, equal_nan=True)
    assert np.array_equal(fd, S.flags)
