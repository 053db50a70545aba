"""The budget of residual evaluations of the common u2p pass: any value that
set_tune takes, up to the largest, bounds what it says.  A large one leaves no
point (and no cell of a grid) to the deferred pass that no bound would not."""
import os
import subprocess

import numpy as np
import pytest

from koral_amd import params as KP, problems as PR, grid as GR

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OVER = -200
LARGE = [1 << 27, (1 << 28) - 1, 1 << 28, 1 << 30, (1 << 31) - 1]


def test_host_budgets(oracle, tmp_path):
    exe = tmp_path / "u2p_budget_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                    "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I",
                    os.path.join(ROOT, "koral_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "host", "u2p_budget_check.cpp"), "-o", str(exe)], check=True)
    P = KP.params_torus_mhd()
    n = 3000
    pp, guess, g20, G20 = PR.u2p_guess_states(P, n, seed=3)
    uu = oracle.p2u(P, pp, g20, G20)
    uu[::9, 1] *= 0.5  # some that the hot inversion gives up on
    inp, out = tmp_path / "in.bin", tmp_path / "out.bin"
    with open(inp, "wb") as f:
        f.write(bytes(P))
        f.write(np.int64(n).tobytes())
        for a in (guess, uu, g20, G20):
            f.write(np.ascontiguousarray(a, dtype=np.float64).tobytes())

    def run(budget):
        subprocess.run([str(exe), str(inp), str(budget), str(out)], check=True)
        return np.fromfile(out, np.int32)
    free = run(0)
    assert np.all(free != OVER) and np.any(free < 0)
    over = [(run(b) == OVER).sum() for b in (1, 2, 4, 8, 32)]
    assert over[0] > 0 and over == sorted(over, reverse=True)
    for b in LARGE:
        assert np.array_equal(run(b), free), b


@pytest.mark.gpu
@pytest.mark.parametrize("budget", [LARGE[0], LARGE[-1]])
def test_gpu_grid_large_budget(budget):
    from koral_amd.gridrun import DeviceGrid
    P = KP.params_torus_mhd()
    spec, p = PR.torus_setup(P, n=(16, 16, 8))
    runs = []
    for b in (0, budget):
        dg = DeviceGrid(P, spec)
        t = dg.get_tune()
        t.u2p_budget = b
        dg.set_tune(t)
        assert dg.get_tune().u2p_budget == b
        dg.upload(GR.to_aos(p))
        dg.init()
        dg.run(2)
        runs.append((dg.deferred_counts()[3],) + dg.download())
    assert runs[0][0] == runs[1][0]
    for a, b in zip(runs[0][1:], runs[1][1:]):
        assert np.array_equal(a, b, equal_nan=True)
