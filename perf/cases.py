"""Workloads of the framework through its public entry points, for timing and
for comparing the outputs of two builds.

A case is a dict of plain values; `kind` names the path:

  u2p       batched primitive inversion (koral_amd.cell.u2p) from a stale guess
  implicit  batched implicit gas-radiation solve (koral_amd.cell.implicit)
  learned   the same solve from network starts (koral_amd.learn.implicit_learned)
  infer     network inference over many cells (koral_amd.learn.Net.infer)
  fit       one epoch of network training (koral_amd.learn.Net.fit)
  tube      RK2IMEX steps of the 1-D radiation shock tube (DeviceGrid.run)
  torus     RK2IMEX steps of the GRMHD torus (DeviceGrid.run)
  ops       op_explicit followed by calc_u2p on the GRMHD torus, the calls a
            host program makes when it keeps its own step loop

Points of the batched paths are drawn on the device: half or more on
Kerr-Schild (spin 0.9), the rest in flat space.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from koral_amd import cell, learn, params as KP, problems as PR, grid as GR
from koral_amd._lib import check
from koral_amd.gridrun import DeviceGrid

DEV = "cuda"
F64 = torch.float64


def listed():
    return [
        # a handful of cells a host code hands over between its own operators: launch latency
        {"name": "u2p_mhd_1k", "kind": "u2p", "n": 1009, "rad": 0},
        # a whole GRMHD tile inverted at once
        {"name": "u2p_mhd_1m", "kind": "u2p", "n": 1 << 20, "rad": 0},
        # field + radiation layout, odd size
        {"name": "u2p_m1_200k", "kind": "u2p", "n": 200003, "rad": 1},
        # the implicit source of a small tile: too few cells to fill the chip
        {"name": "implicit_3k", "kind": "implicit", "n": 3001},
        # the batched implicit solve at its benchmark size
        {"name": "implicit_4m", "kind": "implicit", "n": 1 << 22},
        # the same solve from the learned starts, weights kept by the program
        {"name": "learned_250k", "kind": "learned", "n": 250007},
        # starts of a whole batch from one network
        {"name": "infer_1m", "kind": "infer", "n": 1 << 20},
        # training the networks: one epoch over 16 mini-batches
        {"name": "fit_16x4096", "kind": "fit", "batch": 4096, "batches": 16},
        # 1-D tube at its benchmark size, the smallest grid: launches dominate
        {"name": "tube_512", "kind": "tube", "nx": 512, "steps": 20, "graph": True},
        # the default benchmark grid from its initial state, replayed as a graph
        {"name": "torus_128x128x64", "kind": "torus", "nx": 128, "ny": 128, "nz": 64, "advance": 0, "steps": 2,
         "graph": True},
        # the largest configured grid, after the torus has developed its rare cells
        {"name": "torus_192x192x96_late", "kind": "torus", "nx": 192, "ny": 192, "nz": 96, "advance": 40, "steps": 1,
         "graph": True},
        # a ragged tile driven operator by operator
        {"name": "ops_95x66x37", "kind": "ops", "nx": 95, "ny": 66, "nz": 37, "advance": 4},
    ]


def draw(rng):
    def lu(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    kind = rng.choice(["u2p", "u2p", "implicit", "implicit", "learned", "infer", "fit", "tube", "torus", "torus",
                       "ops"])
    if kind == "u2p":
        return {"kind": kind, "n": lu(500, 1 << 20), "rad": rng.randint(0, 1)}
    if kind == "implicit":
        return {"kind": kind, "n": lu(1000, 1 << 21)}
    if kind == "learned":
        return {"kind": kind, "n": lu(2000, 1 << 18)}
    if kind == "infer":
        return {"kind": kind, "n": lu(500, 1 << 21)}
    if kind == "fit":
        return {"kind": kind, "batch": rng.randint(500, 4096), "batches": rng.randint(4, 16)}
    if kind == "tube":
        return {"kind": kind, "nx": lu(100, 4000), "steps": rng.randint(5, 30), "graph": bool(rng.randint(0, 1))}
    nx, ny, nz = lu(24, 160), lu(16, 144), rng.choice([1, lu(8, 80), lu(8, 80)])
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "advance": rng.randint(0, 30)}
    if kind == "torus":
        c.update(steps=rng.randint(1, 2), graph=bool(rng.randint(0, 1)))
    return c


# ---------------------------------------------------------------------------
# points of the batched paths
# ---------------------------------------------------------------------------
def _rng(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uni(g, n, a, b):
    return a + (b - a) * torch.rand(n, generator=g, device=DEV, dtype=F64)


def _loguni(g, n, a, b):
    return torch.exp(_uni(g, n, math.log(a), math.log(b)))


def _metric(g, n, ks_fraction, rmin, cmax, spin=0.9):
    """g20, G20 [20][n] (rows of 4x5: the 4x4 metric, then a column whose last
    entry is sqrt(-g) or g_tt + 1): Kerr-Schild closed forms, or flat."""
    ks = _uni(g, n, 0., 1.) < ks_fraction
    r, c = _uni(g, n, rmin, 50.), _uni(g, n, -cmax, cmax)
    s2 = 1. - c * c
    a = spin
    sig = r * r + a * a * c * c
    h = 2. * r / sig
    z = torch.zeros_like(r)
    one = torch.ones_like(r)
    lo = torch.stack([
        -1. + h, h, z, -a * h * s2, z,
        h, 1. + h, z, -a * s2 * (1. + h), z,
        z, z, sig, z, z,
        -a * h * s2, -a * s2 * (1. + h), z, s2 * (sig + a * a * s2 * (1. + h)), sig * torch.sqrt(s2)])
    up = torch.stack([
        -1. - h, h, z, z, z,
        h, (r * r - 2. * r + a * a) / sig, z, a / sig, z,
        z, z, 1. / sig, z, z,
        z, a / sig, z, 1. / (sig * s2), h])
    flo = torch.stack([-one, z, z, z, z, z, one, z, z, z, z, z, one, z, z, z, z, z, one, one])
    fup = torch.stack([-one, z, z, z, z, z, one, z, z, z, z, z, one, z, z, z, z, z, one, z])
    return torch.where(ks, lo, flo).contiguous(), torch.where(ks, up, fup).contiguous()


def _relvel(g, n, lo, gamma):
    """Velocities relative to the normal observer with Lorentz factor gamma in
    random directions: u = sqrt(gamma^2 - 1) L^-T d with g_ij = L L^T."""
    d = torch.randn((3, n), generator=g, device=DEV, dtype=F64)
    d = d / torch.sqrt((d * d).sum(0))
    g11, g12, g13, g22, g23, g33 = lo[6], lo[7], lo[8], lo[12], lo[13], lo[18]
    l11 = torch.sqrt(g11)
    l21, l31 = g12 / l11, g13 / l11
    l22 = torch.sqrt(g22 - l21 * l21)
    l32 = (g23 - l31 * l21) / l22
    l33 = torch.sqrt(g33 - l31 * l31 - l32 * l32)
    z = d[2] / l33
    y = (d[1] - l32 * z) / l22
    x = (d[0] - l21 * y - l31 * z) / l11
    return torch.sqrt(gamma * gamma - 1.) * torch.stack([x, y, z])


def _entropy(gamma, rho, u):
    k = 1. / (gamma - 1.)
    return rho * (k * torch.log((gamma - 1.) * u) - (k + 1.) * torch.log(rho))


def _u2p_points(P, n, seed, nv, ee):
    """True primitives, and the guess a time step leaves behind."""
    g = _rng(seed)
    lo, up = _metric(g, n, 0.7, 2., 0.98)
    rho = _loguni(g, n, 1e-4, 1e1)
    u = rho * _loguni(g, n, 1e-4, 1e1)
    true = torch.zeros((nv, n), device=DEV, dtype=F64)
    true[0], true[1] = rho, u
    true[2:5] = _relvel(g, n, lo, _uni(g, n, 1., 5.))
    true[5] = _entropy(P.gamma, rho, u)
    pmag = (P.gamma - 1.) * u / _loguni(g, n, 1., 1e3)
    true[6:9] = _relvel(g, n, lo, torch.sqrt(1. + 2. * pmag))
    if nv > 9:
        true[ee] = u * _loguni(g, n, 1e-3, 1e3)
        true[ee + 1:ee + 4] = _relvel(g, n, lo, _uni(g, n, 1., 5.))
    s = _loguni(g, n, 1e-4, 0.1)
    guess = true.clone()
    for k in (0, 1):
        guess[k] *= torch.exp(s * torch.randn(n, generator=g, device=DEV, dtype=F64))
    vmag = torch.sqrt((true[2:5] ** 2).sum(0)) + 0.1
    guess[2:5] += s * vmag * torch.randn((3, n), generator=g, device=DEV, dtype=F64)
    return true, guess, lo, up


def _implicit_points(P, n, seed):
    """The batched solve's distribution (problems.implicit_batch_states)."""
    g = _rng(seed)
    lo, up = _metric(g, n, 0.5, 3., 0.95)
    ee = P.ee
    rho, T = _loguni(g, n, 1e-6, 1e2), _loguni(g, n, 1e4, 1e9)
    u = KP.u_from_Trho(P, T, rho)
    pp = torch.zeros((P.nv, n), device=DEV, dtype=F64)
    pp[0], pp[1] = rho, u
    pp[2:5] = _relvel(g, n, lo, _uni(g, n, 1., 10.))
    pp[5] = _entropy(P.gamma, rho, u)
    pp[ee] = u * _loguni(g, n, 1e-4, 1e4)
    pp[ee + 1:ee + 4] = _relvel(g, n, lo, _uni(g, n, 1., 10.))
    rhocgs = rho / P.ggg * P.ccc * P.ccc / P.masscm / P.masscm
    kappa = P.kappa_a_coef * rhocgs / T ** 3.5 / P.ggg * P.ccc * P.ccc / P.masscm * rho
    return pp, lo, up, _loguni(g, n, 1e-3, 1e6) / kappa


# ---------------------------------------------------------------------------
# the network in 64 bits (training of the kept weights, exact values)
# ---------------------------------------------------------------------------
SHAPES = ((learn.NH, learn.NIN), (learn.NH, learn.NH), (learn.NH, learn.NH), (learn.NOUT, learn.NH))


def _theta0(seed):
    """He-style uniform weights and zero biases, flat, float64 on the device."""
    rng = np.random.default_rng(seed)
    parts = []
    for o, i in SHAPES:
        lim = math.sqrt(6. / i)
        parts += [rng.uniform(-lim, lim, o * i), np.zeros(o)]
    return torch.from_numpy(np.concatenate(parts).astype(np.float32)).to(DEV, F64)


def _net(theta, X):
    a, k = X, 0
    for layer, (o, i) in enumerate(SHAPES):
        z = theta[k:k + o * i].view(o, i) @ a + theta[k + o * i:k + o * i + o, None]
        k += o * i + o
        a = torch.nn.functional.gelu(z, approximate="tanh") if layer < 3 else z
    return a


class _Adam:
    def __init__(self, theta):
        self.th = theta.clone().requires_grad_(True)
        self.m, self.v, self.k = torch.zeros_like(theta), torch.zeros_like(theta), 0

    def step(self, X, T, lr):
        loss = ((_net(self.th, X) - T) ** 2).mean()
        g, = torch.autograd.grad(loss, self.th)
        self.k += 1
        self.m = 0.9 * self.m + 0.1 * g
        self.v = 0.999 * self.v + 0.001 * g * g
        mh, vh = self.m / (1. - 0.9 ** self.k), self.v / (1. - 0.999 ** self.k)
        self.th.data -= lr * mh / (torch.sqrt(vh) + 1e-8)
        return float(loss.detach())


def _fit64(opt, X, T, batch, lr, seed):
    """One epoch over the mini-batches Net.fit takes with this seed."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    perm = torch.randperm(X.shape[1], device=DEV, generator=gen)
    losses = []
    for k, b in enumerate(range(0, X.shape[1] - batch + 1, batch)):
        idx = perm[b:b + batch]
        losses.append(opt.step(X[:, idx].double(), T[:, idx].double(), lr))
    return [float(np.mean(losses[::64]))]


@functools.lru_cache(maxsize=1)
def _kept_nets():
    """Gas and radiation networks trained on plain solves, as a program that
    uses the learned solve keeps them: (theta, norm) of each."""
    P = KP.params_implicit_batch()
    pp0, lo, up, dt = _implicit_points(P, 1 << 16, 4321)
    uu, pp1 = cell.p2u(P, pp0, lo, up), pp0.clone()
    _, info = cell.implicit(P, uu, pp1, lo, up, dt)
    F, Tg, Tr = learn.training_pairs(P, pp0, pp1, dt, info)
    nets = []
    for T in (Tg, Tr):
        norm = learn.normalisation(F, T)
        X, Y = (x.double() for x in learn.standardise(F, T, norm))
        opt = _Adam(_theta0(1))
        for k in range(600):
            b = (k * 2048) % (X.shape[1] - 2048)
            opt.step(X[:, b:b + 2048], Y[:, b:b + 2048], 2e-3 if k < 300 else 5e-4)
        nets.append((opt.th.detach().float().cpu().numpy(), norm))
    return nets


def _pairs(n, seed):
    """Standardised features and smooth targets with scatter."""
    g = _rng(seed)
    X = torch.randn((learn.NIN, n), generator=g, device=DEV)
    W = torch.randn((learn.NOUT, learn.NIN), generator=_rng(77), device=DEV) * 0.5
    T = torch.sin(W @ X) + 0.3 * X[:learn.NOUT] + 0.1 * torch.randn((learn.NOUT, n), generator=g, device=DEV)
    return X.contiguous(), T.contiguous()


# ---------------------------------------------------------------------------
# grids
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _torus_base(nx, ny, nz):
    return PR.torus_setup(KP.params_torus_mhd(), n=(nx, ny, nz), pert=0.)


@functools.lru_cache(maxsize=4)
def _tube_base(nx):
    return PR.tube_setup(KP.params_tube(), nx=nx)


class _View:
    """Device memory of a grid; holds the grid, which owns it."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (ptr, False), "version": 2}


def _views(dg):
    """The grid's resident state (koral_hip_grid_device_state) as tensors."""
    p, u = ctypes.c_void_p(), ctypes.c_void_p()
    check(dg.L.koral_hip_grid_device_state(dg.h, ctypes.byref(p), ctypes.byref(u), None), "device_state")
    shape = (dg.P.nv,) + tuple(dg.spec.shape)
    views = [torch.as_tensor(_View(dg, x.value, shape), device=DEV) for x in (p, u)]
    for v in views:
        v.grid = dg  # the memory lives as long as the tensor does
    return views


def _prepare_grid(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "tube":
        P = KP.params_tube()
        spec, p = _tube_base(case["nx"])
        p = p.copy()
        p[0] *= 1. + 1e-3 * rng.uniform(-1., 1., p[0].shape)
    else:
        P = KP.params_torus_mhd()
        spec, p = _torus_base(case["nx"], case["ny"], case["nz"])
        p = p.copy()
    p[1] *= 1. + 0.02 * rng.uniform(-1., 1., p[1].shape)
    stream = torch.cuda.Stream()
    dg = DeviceGrid(P, spec, stream=stream.cuda_stream)
    dg.upload(GR.to_aos(p))
    dg.init()
    if case.get("advance"):
        dg.run(case["advance"])
    if case.get("graph"):
        dg.use_graph(True)
    stream.synchronize()
    vp, vu = _views(dg)
    return {"case": case, "dg": dg, "stream": stream, "p": vp, "u": vu, "p0": vp.clone(), "u0": vu.clone(),
            "t": dg.t, "dt": dg.dt}


def _run_grid(s):
    """From the kept state: the steps (or the two operators), to the state."""
    dg, case = s["dg"], s["case"]
    with torch.cuda.stream(s["stream"]):
        s["p"].copy_(s["p0"])
        s["u"].copy_(s["u0"])
    dg.t, dg.dt = s["t"], s["dt"]
    if case["kind"] == "ops":
        tsd = dg.explicit(dg.t, dg.dt)
        dg.u2p()
        torch.cuda.current_stream().wait_stream(s["stream"])
        return {"p": s["p"], "u": s["u"], "tsd": tsd}
    dg.run(case["steps"])
    return {"p": s["p"], "u": s["u"], "t": dg.t, "dt": dg.dt, "counters": dg.counters.copy()}


# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "u2p":
        P = KP.params_implicit_batch() if case["rad"] else KP.params_torus_mhd()
        true, guess, lo, up = _u2p_points(P, case["n"], seed, P.nv, P.ee)
        return {"case": case, "P": P, "uu": cell.p2u(P, true, lo, up), "pp": guess, "g": lo, "G": up}
    if kind in ("implicit", "learned"):
        P = KP.params_implicit_batch()
        pp, lo, up, dt = _implicit_points(P, case["n"], seed)
        s = {"case": case, "P": P, "uu": cell.p2u(P, pp, lo, up), "pp": pp, "g": lo, "G": up, "dt": dt}
        if kind == "learned":
            s["nets"] = [learn.Net(kind=k, theta=th, norm=nm)
                         for k, (th, nm) in zip((learn.GAS, learn.RAD), _kept_nets())]
        return s
    if kind == "infer":
        X, _ = _pairs(case["n"], seed)
        return {"case": case, "X": X, "net": learn.Net(theta=_theta0(3).cpu().numpy())}
    if kind == "fit":
        X, T = _pairs(case["batch"] * case["batches"], seed)
        net = learn.Net(theta=_theta0(3).cpu().numpy())
        net.fit(X, T, epochs=1, lr=0., batch=case["batch"], seed=1)  # settled Adam moments, as in mid-training
        return {"case": case, "X": X, "T": T, "net": net}
    return _prepare_grid(case, seed)


def run(s):
    kind = s["case"]["kind"]
    if kind == "u2p":
        uu, pp = s["uu"].clone(), s["pp"].clone()
        ret, flags = cell.u2p(s["P"], uu, pp, s["g"], s["G"])
        return {"uu": uu, "pp": pp, "ret": ret, "flags": flags}
    if kind == "implicit":
        uu, pp = s["uu"].clone(), s["pp"].clone()
        flags, info = cell.implicit(s["P"], uu, pp, s["g"], s["G"], s["dt"])
        return {"uu": uu, "pp": pp, "flags": flags, "info": info}
    if kind == "learned":
        uu, pp = s["uu"].clone(), s["pp"].clone()
        flags, info = learn.implicit_learned(s["P"], s["nets"][0], s["nets"][1], uu, pp, s["g"], s["G"], s["dt"],
                                             maxiter=16)
        return {"uu": uu, "pp": pp, "flags": flags, "info": info}
    if kind == "infer":
        return s["net"].infer(s["X"])
    if kind == "fit":
        hist = s["net"].fit(s["X"], s["T"], epochs=1, lr=1e-3, batch=s["case"]["batch"], seed=2)
        return {"loss": torch.tensor(hist), "theta": s["net"].get()[0]}
    return _run_grid(s)


def work(case):
    """Inputs read once and outputs written once; FP64 or matrix operations
    the path's algorithm needs."""
    kind = case["kind"]
    if kind == "u2p":
        nv = 13 if case["rad"] else 9
        return {"bytes": case["n"] * (8. * (4 * nv + 40) + 32.), "flops": case["n"] * 1500.}
    if kind in ("implicit", "learned"):
        return {"bytes": case["n"] * (8. * (4 * 13 + 41) + 52.), "flops": case["n"] * 627940.}
    if kind == "infer":
        return {"bytes": case["n"] * 4. * (learn.NIN + learn.NOUT), "flops": case["n"] * 2. * 34688}
    if kind == "fit":
        n = float(case["batch"] * case["batches"])
        return {"bytes": n * 4. * 15 + case["batches"] * 6. * 4 * 35076, "flops": n * 6. * 34688}
    if kind == "tube":
        return {"bytes": 1. * case["nx"] * case["steps"] * 2004., "flops": 1. * case["nx"] * case["steps"] * 2e5}
    zones = float(case["nx"] * case["ny"] * case["nz"])
    if kind == "ops":
        return {"bytes": zones * 8. * 4 * 9, "flops": zones * 11000.}
    return {"bytes": zones * case["steps"] * 8. * 4 * 9, "flops": zones * case["steps"] * 24814.}


def exact(case, seed):
    """64-bit values where a closed form or plain torch gives them: the
    primitives an inversion has to find, the network's outputs and one epoch of
    its training.  The implicit solve and the grid steps have none."""
    kind = case["kind"]
    if kind == "u2p":
        P = KP.params_implicit_batch() if case["rad"] else KP.params_torus_mhd()
        true = _u2p_points(P, case["n"], seed, P.nv, P.ee)[0]
        return {"uu": None, "pp": true, "ret": None, "flags": None}
    if kind == "infer":
        X, _ = _pairs(case["n"], seed)
        th = _theta0(3)
        return torch.cat([_net(th, x.double()) for x in X.split(1 << 18, dim=1)], 1)
    if kind == "fit":
        X, T = _pairs(case["batch"] * case["batches"], seed)
        opt = _Adam(_theta0(3))
        _fit64(opt, X, T, case["batch"], 0., 1)
        hist = _fit64(opt, X, T, case["batch"], 1e-3, 2)
        return {"loss": torch.tensor(hist, dtype=F64), "theta": opt.th.detach()}
    return None
