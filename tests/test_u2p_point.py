"""The batched u2p on points that leave its common path: the b^2/rho floor, the
entropy inversion, negative densities, and both at once.  On the host the
per-point function gives the oracle's result bit for bit and reads the state of
a point at the b^2/rho floor once (its inversion is not run a second time); on
the GPU the kernel does on batches that mix all kinds within a wave."""
import os
import subprocess

import numpy as np
import pytest

from koral_amd import params as KP, problems as PR

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LAYOUTS = [(0, 0), (1, 0), (0, 1), (1, 1)]


def _params(mag, rad):
    P = KP.params_implicit_batch()
    P.mag, P.rad = mag, rad
    P.nv = 6 + 3 * mag + 4 * rad
    return P


def _points(oracle, P, n, seed):
    """True states whose kind is drawn per point, the guess beside them, and
    which points have b^2/2 far above the limit of 100 rho."""
    rng = np.random.default_rng(seed)
    pp, g20, G20 = PR.random_mhd_states(P, n, seed=seed)
    kind = rng.integers(0, 8, n)
    floor = (kind == 1) | (kind == 2) if P.mag else np.zeros(n, bool)
    if P.mag:
        B2 = (pp[:, 6:9] ** 2).sum(1)
        # the lab field bounds b^2 from below by its square over gamma^2 <= 25
        pp[floor, 6:9] *= np.sqrt(25. * 1000. * pp[floor, 0] / B2[floor])[:, None]
    uu = oracle.p2u(P, pp, g20, G20)
    bad = (kind == 2) | (kind == 3)
    uu[bad, 1] *= 0.5
    uu[kind == 4, 0] *= -1.
    guess = pp.copy()
    s = np.exp(rng.uniform(np.log(1e-4), np.log(0.1), n))
    guess[:, 0] *= np.exp(s * rng.standard_normal(n))
    guess[:, 1] *= np.exp(s * rng.standard_normal(n))
    return uu, guess, g20, G20, floor


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("up") / "u2p_point_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fopenmp", "-ffp-contract=off", "-fno-fast-math", "-I",
                    os.path.join(ROOT, "koral_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "host", "u2p_point_check.cpp"), "-o", str(out)], check=True)
    return str(out)


@pytest.mark.parametrize("mag,rad", LAYOUTS)
def test_host_points(oracle, exe, tmp_path, mag, rad):
    P = _params(mag, rad)
    n = 20000
    uu, guess, g20, G20, floor = _points(oracle, P, n, seed=11 + mag + 2 * rad)
    inp, out = tmp_path / "batch.bin", tmp_path / "out.bin"
    with open(inp, "wb") as f:
        f.write(bytes(P))
        f.write(np.int64(n).tobytes())
        for a in (guess, uu, g20, G20):
            f.write(np.ascontiguousarray(a, dtype=np.float64).tobytes())
    subprocess.run([exe, str(inp), str(out)], check=True)
    raw = np.fromfile(out, np.uint8)
    m = 8 * P.nv * n
    ph = raw[:m].view(np.float64).reshape(n, P.nv)
    uh = raw[m:2 * m].view(np.float64).reshape(n, P.nv)
    oh = raw[2 * m:].view(np.int32).reshape(n, 7)
    uo, po, ro, fo = oracle.u2p(P, uu, guess, g20, G20)
    assert np.array_equal(ph, po, equal_nan=True) and np.array_equal(uh, uo, equal_nan=True)
    assert np.array_equal(oh[:, 0], ro)
    assert np.array_equal(oh[:, 1:5], fo[:, [0, 4, 2, 3]])
    _, hot = oracle.u2p_solver(P, uu, guess, g20, G20, 0)
    once = (hot >= 0) & (uu[:, 0] >= 0.)
    floored = once & floor
    assert np.all(oh[once, 5] == 1) and np.any(oh[:, 5] == 2)
    # the rare path reads the metric again
    assert np.all(oh[floored, 6] == 2) and (not mag or floored.sum() > n // 16)


@pytest.mark.gpu
@pytest.mark.parametrize("mag,rad", LAYOUTS)
@pytest.mark.parametrize("n", [1, 63, 257, 5003])
def test_gpu_points(oracle, mag, rad, n):
    from koral_amd import cell
    P = _params(mag, rad)
    uu, guess, g20, G20, _ = _points(oracle, P, n, seed=23 + n + mag + 2 * rad)
    U, Q, g, G = (cell.to_dev(x) for x in (uu, guess, g20, G20))
    ret, flags = cell.u2p(P, U, Q, g, G)
    uo, po, ro, fo = oracle.u2p(P, uu, guess, g20, G20)
    assert np.array_equal(cell.to_host(Q), po, equal_nan=True)
    assert np.array_equal(cell.to_host(U), uo, equal_nan=True)
    assert np.array_equal(ret.cpu().numpy(), ro)
    assert np.array_equal(flags.cpu().numpy().T, fo)
