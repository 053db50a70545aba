"""The batched implicit solve at the edges of its schedules: a single cell, a
ragged wave, the largest batch of the wave-per-cell chain and the first of the
per-attempt passes, and metrics whose two halves differ in the last bit (which
take the passes' general variant).  Device against oracle, identical bit for
bit: state, flags, attempts and iterations."""
import numpy as np
import pytest

from koral_amd import params as KP, problems as PR

pytestmark = pytest.mark.gpu

LAST_WAVE = 1 << 14  # IMP_WAVE_CELLS


def _solve(oracle, n, asym, starts=False):
    import torch
    from koral_amd import cell, learn as LN
    P = KP.params_implicit_batch()
    pp, g20, G20, dt = PR.implicit_batch_states(P, n, seed=n)
    if asym:
        # one ulp on the lower half of a few cells' metrics
        for k in (4 * 1 + 1, 5 * 1, 5 * 3 + 1):
            for a in (g20, G20):
                a[:: 7, k] = np.nextafter(a[:: 7, k], 2. * a[:: 7, k])
    uu = oracle.p2u(P, pp, g20, G20)
    U, Pp, g, G = (cell.to_dev(x) for x in (uu, pp, g20, G20))
    dtd = torch.from_numpy(dt).cuda()
    ee = P.ee
    if starts:
        rng = np.random.default_rng(n)
        gx = pp[:, 1:5] * (1. + 0.1 * rng.standard_normal((n, 4)))
        gxr = pp[:, ee:ee + 4] * (1. + 0.1 * rng.standard_normal((n, 4)))
        gx[:, 0], gxr[:, 0] = np.abs(gx[:, 0]), np.abs(gxr[:, 0])
        gx[::5, 0] = np.nan  # no learned try
        fl, info = LN.implicit_from(P, cell.to_dev(gx), cell.to_dev(gxr), U, Pp, g, G, dtd, maxiter=16)
        ref = oracle.implicit(P, uu, pp, g20, G20, dt, nthreads=8, gx=gx, gxr=gxr, maxiter=16)
    else:
        fl, info = cell.implicit(P, U, Pp, g, G, dtd)
        ref = oracle.implicit(P, uu, pp, g20, G20, dt, nthreads=8)
    uo, po, flo, io = ref
    assert np.array_equal(info.cpu().numpy().T, io)
    assert np.array_equal(cell.to_host(Pp), po, equal_nan=True)
    assert np.array_equal(cell.to_host(U), uo, equal_nan=True)
    assert np.array_equal(fl.cpu().numpy().T, flo)


@pytest.mark.parametrize("n", [1, 7, 65, 1025, LAST_WAVE, LAST_WAVE + 1, 20011])
def test_sizes(oracle, n):
    _solve(oracle, n, False)


@pytest.mark.parametrize("n", [129, LAST_WAVE + 9])
def test_asymmetric_metric(oracle, n):
    _solve(oracle, n, True)


@pytest.mark.parametrize("n", [65, LAST_WAVE + 65])
def test_given_starts(oracle, n):
    _solve(oracle, n, False, starts=True)
