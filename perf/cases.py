"""The work that a user of this library has it do, as cases that can be timed and checked.

A case is a dict of plain values; ``listed()`` gives the fixed ones, ``draw(rng)`` one
more of the same ranges, ``prepare(case, seed)`` the inputs and the plan a program holds
before the call, ``run(state)`` one pass through the public API, ``work(case)`` the bytes
and operations of a pass, and ``exact(case, seed)`` the outputs as plain FP64 direct sums
(torch), without this library.

The kinds:

* ``host``    the host API on numpy arrays with its defaults (FP64, dense class M2L):
              ``FMM``, ``build_expansions``, ``evaluate_at_sources``; small problems, where
              the plan and the launches count.
* ``replay``  a captured pass sequence replayed with new charges (an inner loop on a small
              fixed geometry).
* ``matvec``  one matvec on a kept plan (an iterative solver on a fixed geometry).
* ``solve``   a whole solve from device-resident points: plan, expansions, outputs at the
              sources and, where ``nt`` > 0, potential and gradient at targets (moving points).
* ``field``   a whole solve of a large source set whose field is wanted at fewer targets.
* ``stokes_api``  the Stokes front end on host arrays (``StokesFMMPlan``, ``stokes_fmm_eval_``).
* ``circle``  the 2D circle method on a kept plan: potential at the sources and at targets.
* ``served``  a burst of host requests through a ``Server`` with four slots.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "flexiblefmm.jl_amd"))

import ffmm  # noqa: E402
from ffmm.serving import Server  # noqa: E402

BOX3 = (np.zeros(3), 1.0)
BOX2 = ((0.0, 0.0), 1.0)
KAPPA = 5.0          # the Yukawa parameter of the served stream
DEV = "cuda:0"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(name, kind, method, n, **kw):
    c = dict(kind=kind, method=method, n=n, nt=0, p=8, ppl=64, layout="mixture", precision="mixed", m2l="spectral")
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the first thing a new user runs: host arrays, every default
        _case("host_4k", "host", "cube", 4000, ppl=50, layout="mixed", precision="f64", m2l="dense"),
        # an inner loop on a small fixed geometry: launches are what it pays for
        _case("replay_10k", "replay", "cube", 10_000, layout="uniform"),
        # the reference's published CPU case, FP64 with the default class M2L, on a kept plan
        _case("matvec_100k_f64_dense", "matvec", "cube", 100_000, ppl=200, layout="uniform", precision="f64", m2l="dense"),
        # a middle-sized FP64 solve with the spectral M2L, outputs at sources and targets
        _case("solve_300k_f64", "solve", "cube", 300_007, nt=100_003, precision="f64"),
        # the headline workload's form (mixed precision, moving points) at a quarter of its size
        _case("solve_1m_mixed", "solve", "cube", 1_000_000, nt=250_000),
        # the headline workload's sources; the field at fewer targets
        _case("field_4m_mixed", "field", "cube", 4_000_000, nt=150_000),
        # the served Yukawa requests
        _case("yukawa_200k_mixed", "solve", "yukawa", 200_000, p=10, m2l="dense"),
        # boundary integral points: stokeslets and stresslets on 64 ellipsoids
        _case("stokes_250k_mixed", "solve", "stokes", 250_000, p=10, layout="ellipsoids", m2l="dense"),
        # the same at a larger size, the velocity at probe points in the fluid
        _case("stokes_field_1m_mixed", "field", "stokes", 1_000_000, nt=40_000, p=10, layout="ellipsoids", m2l="dense"),
        # the Stokes front end as the reference's users call it (FP64, its defaults but p)
        _case("stokes_api_20k", "stokes_api", "stokes", 20_011, p=10, ppl=200, layout="ellipsoids", precision="f64",
              m2l="dense"),
        # 2D, FP64: the circle configuration
        _case("circle_100k", "circle", "circle", 100_000, nt=50_000, p=60, ppl=50, layout="uniform", precision="f64",
              m2l="dense"),
        # a burst of mixed requests through the server
        _case("served_10", "served", "mix", 60_000, nt=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "replay", "matvec", "solve_f64", "solve_mixed", "solve_mixed", "field", "yukawa",
                       "laplace", "stokes", "stokes_field", "stokes_api", "circle", "served"])
    lay = rng.choice(["uniform", "mixture", "mixed"])
    if kind == "host":
        return _case("", "host", "cube", _log(rng, 300, 30_000), ppl=rng.choice([30, 50, 100]), layout=lay,
                     precision="f64", m2l="dense")
    if kind == "replay":
        return _case("", "replay", "cube", _log(rng, 2000, 60_000), ppl=rng.choice([50, 64, 100]), layout=lay)
    if kind == "matvec":
        return _case("", "matvec", "cube", _log(rng, 10_000, 200_000), p=rng.choice([6, 8, 8]), layout=lay,
                     ppl=rng.choice([64, 100, 200]), precision="f64", m2l="dense")
    if kind == "solve_f64":
        n = _log(rng, 20_000, 400_000)
        return _case("", "solve", "cube", n, nt=rng.choice([0, n // 3 + 1]), layout=lay, ppl=rng.choice([64, 100]),
                     precision="f64")
    if kind == "solve_mixed":
        n = _log(rng, 10_000, 1_000_000)
        return _case("", "solve", "cube", n, nt=rng.choice([0, n // 4 + 1]), layout=lay,
                     ppl=rng.choice([50, 64, 100, 150]))
    if kind == "field":
        return _case("", "field", "cube", _log(rng, 500_000, 3_500_000), nt=_log(rng, 10_000, 150_000), layout=lay,
                     ppl=rng.choice([64, 100]))
    if kind == "yukawa":
        return _case("", "solve", "yukawa", _log(rng, 5000, 250_000), p=10, layout=lay, m2l="dense",
                     precision=rng.choice(["mixed", "mixed", "f64"]))
    if kind == "laplace":   # charges and dipoles, the spherical-harmonic method
        return _case("", "matvec", "dipole", _log(rng, 3000, 80_000), p=rng.choice([8, 10]), layout=lay, m2l="dense",
                     precision=rng.choice(["mixed", "f64"]))
    if kind == "stokes":
        return _case("", "solve", "stokes", _log(rng, 10_000, 250_000), p=rng.choice([8, 10]), layout="ellipsoids",
                     ppl=rng.choice([64, 100]), m2l="dense", precision=rng.choice(["mixed", "mixed", "f64"]))
    if kind == "stokes_field":
        return _case("", "field", "stokes", _log(rng, 200_000, 900_000), nt=_log(rng, 5000, 40_000), p=10,
                     layout="ellipsoids", m2l="dense")
    if kind == "stokes_api":
        return _case("", "stokes_api", "stokes", _log(rng, 1000, 30_000), p=rng.choice([8, 10]), ppl=200,
                     layout="ellipsoids", precision="f64", m2l="dense")
    if kind == "circle":
        n = _log(rng, 5000, 300_000)
        return _case("", "circle", "circle", n, nt=n // 2 + 1, p=rng.choice([40, 60]), ppl=50,
                     layout=rng.choice(["uniform", "mixture"]), precision="f64", m2l="dense")
    return _case("", "served", "mix", _log(rng, 15_000, 80_000), nt=rng.randint(4, 12))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, dtype=torch.float64, device=DEV, generator=g)


def _randn(g, *shape):
    return torch.randn(*shape, dtype=torch.float64, device=DEV, generator=g)


def _points(g, n, layout, dim=3):
    """n points in the unit box: uniform; a mixture of 32 Gaussians (centres uniform in
    [0.1, 0.9], sigma log-uniform in [0.005, 0.05]); or half on a sphere, a quarter in a
    tight cluster, the rest uniform (a deep adaptive tree)."""
    if layout == "uniform":
        return _rand(g, n, dim)
    if layout == "mixture":
        cen = 0.1 + 0.8 * _rand(g, 32, dim)
        sig = torch.exp(math.log(0.005) + math.log(10.0) * _rand(g, 32))
        comp = torch.arange(n, device=DEV) % 32
        return (cen[comp] + sig[comp, None] * _randn(g, n, dim)).clamp_(0.0, 1.0)
    ns, nk = n // 2, n // 4
    v = _randn(g, ns, dim)
    s = 0.5 + 0.3 * v / v.norm(dim=1, keepdim=True)
    return torch.cat([s, 0.9 + 0.002 * _randn(g, nk, dim), _rand(g, n - ns - nk, dim)]).clamp_(0.0, 1.0)


def _ellipsoids(g, n, nell=64):
    """n points on 64 ellipsoids (semi-axes uniform in [0.02, 0.08], random rotations),
    area-uniform on each, and their unit normals."""
    cen, axes = 0.15 + 0.7 * _rand(g, nell, 3), 0.02 + 0.06 * _rand(g, nell, 3)
    R = torch.linalg.qr(_randn(g, nell, 3, 3).cpu())[0].to(DEV)
    pts, nrm = [], []
    for e in range(nell):
        m = n // nell + (1 if e < n % nell else 0)
        u = torch.empty((0, 3), dtype=torch.float64, device=DEV)
        while u.shape[0] < m:
            v = _randn(g, 3 * m + 16, 3)
            v = v / v.norm(dim=1, keepdim=True)
            u = torch.cat([u, v[_rand(g, v.shape[0]) < (v / axes[e]).norm(dim=1) * axes[e].min()]])
        u = u[:m]
        w = u / axes[e]
        pts.append(cen[e] + (u * axes[e]) @ R[e].T)
        nrm.append((w / w.norm(dim=1, keepdim=True)) @ R[e].T)
    return torch.cat(pts).clamp_(0.0, 1.0), torch.cat(nrm)


def _inputs(case, seed):
    """points, densities, targets (None when the case has none), on the GPU."""
    g = _gen(seed)
    n, nt, method = case["n"], case["nt"], case["method"]
    if case["layout"] == "ellipsoids":
        x, nrm = _ellipsoids(g, n)
        d = torch.cat([_randn(g, n, 3), _randn(g, n, 3), nrm], 1).contiguous()
    else:
        x = _points(g, n, case["layout"], 2 if method == "circle" else 3)
        d = _randn(g, n, 4) if method == "dipole" else _randn(g, n)
        if method == "dipole":
            d[:, 1:] *= 0.01     # dipoles of the size of the particles that carry them
    t = _rand(g, nt, x.shape[1]) if nt else None
    return x, d, t


def _requests(case, seed):
    """The burst's requests: (kernel, points, charges, geometry key); 70% Laplace on cube
    surfaces, the rest Yukawa, sizes (the case's own) log-uniform from a sixth of n to n,
    every fifth request repeating the first geometry of its kernel with new charges."""
    g, rng = _gen(seed), np.random.default_rng(case["n"])
    first, out = {}, []
    for k in range(case["nt"]):
        lap = k % 10 in (0, 1, 3, 4, 6, 7, 9)
        m = int(np.exp(rng.uniform(np.log(case["n"] / 6), np.log(case["n"]))))
        if k % 5 == 4 and lap in first:
            pts, key = first[lap]
        else:
            pts, key = _points(g, m, "mixture" if rng.random() < 0.5 else "uniform").cpu().numpy(), -1
            if lap not in first:
                key = 2 * (1_000_003 * int(seed) + case["n"]) + int(lap)
                first[lap] = (pts, key)
        out.append((lap, pts, _randn(g, len(pts)).cpu().numpy(), key))
    return out


# what a program keeps for its whole life: the methods with their operator caches, the server
_METHODS = {}
_SERVER = []


def _method(method, p):
    got = _METHODS.get((method, p))
    if got is None:
        if method == "circle":
            m = ffmm.KernelIndependent(ffmm.Laplace2D(), nequiv=p)
            got = (m, ffmm.CircleOperatorCache(m))
        else:
            m = {"cube": lambda: ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=p),
                 "yukawa": lambda: ffmm.SphericalHarmonics(ffmm.Yukawa3D(KAPPA), p=p),
                 "dipole": lambda: ffmm.SphericalHarmonics(ffmm.Laplace3D(), p=p),
                 "stokes": lambda: ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=p)}[method]()
            got = (m, ffmm.OperatorCache(m))
        _METHODS[(method, p)] = got
    return got


def _plan(case, x):
    m, cache = _method(case["method"], case["p"])
    return ffmm.DevicePlan(m, x, ppl=case["ppl"], bbox=BOX3, cache=cache, precision=case["precision"], m2l=case["m2l"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "served":
        if not _SERVER:
            _SERVER.append(Server(nslots=4, hbm_budget=48 << 30))
        return dict(case=case, requests=_requests(case, seed),
                    caches={True: _method("cube", 8)[1], False: _method("yukawa", 10)[1]})
    x, d, t = _inputs(case, seed)
    st = dict(case=case, x=x, d=d, t=t)
    if kind == "host":
        st.update(x=x.cpu().numpy(), d=d.cpu().numpy(), method=_method("cube", 8))
    elif kind == "stokes_api":
        h = d.cpu().numpy()
        m, cache = _method("stokes", case["p"])
        plan = ffmm.StokesFMMPlan(x.cpu().numpy(), p=case["p"], ppl=case["ppl"], bbox=BOX3,
                                  precision=case["precision"])
        st = dict(case=case, plan=plan, f=h[:, 0:3].copy(), g=h[:, 3:6].copy(), nu=h[:, 6:9].copy())
    elif kind == "circle":
        m, cache = _method("circle", case["p"])
        st["plan"] = ffmm.CirclePlan(m, x.cpu().numpy(), ppl=case["ppl"], bbox=BOX2, cache=cache)
    elif kind == "matvec":
        st["plan"] = _plan(case, x)
    elif kind == "replay":
        st["plan"] = _plan(case, x).capture()
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        m, cache = state["method"]
        f = ffmm.FMM(m, state["x"], ppl=case["ppl"], bbox=BOX3, cache=cache)
        st = ffmm.build_expansions(f, state["x"], state["d"])
        return ffmm.evaluate_at_sources(f, st)
    if kind == "replay":
        return state["plan"].replay(state["d"])
    if kind == "matvec":
        if case["method"] == "dipole":
            return state["plan"].matvec(state["d"], ffmm.PotentialGradient)
        return state["plan"].matvec(state["d"])
    if kind == "stokes_api":
        return ffmm.stokes_fmm_eval_(None, state["plan"], stokeslets=state["f"], stresslets=state["g"],
                                     stressvecs=state["nu"])
    if kind == "circle":
        p = state["plan"]
        return [p.matvec(state["d"]), p.evaluate(state["t"])]
    if kind == "served":
        srv = _SERVER[0]
        tickets = [srv.submit(state["caches"][lap], x, q, geometry=key, ppl=64, bbox=BOX3, precision="mixed",
                              m2l="spectral" if lap else "dense") for lap, x, q, key in state["requests"]]
        return [srv.wait(t)[0] for t in tickets]
    plan = _plan(case, state["x"])
    if kind == "field":
        plan.build_expansions(state["d"])
        return plan.evaluate(state["t"], ffmm.Velocity if case["method"] == "stokes" else ffmm.PotentialGradient)
    u = plan.matvec(state["d"])
    if state["t"] is None:
        return u
    return [u, plan.evaluate(state["t"], ffmm.PotentialGradient)]


# ---------------------------------------------------------------------------
# bytes and operations
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the points, densities and outputs once.  Operations: the near field (a leaf
    holds about ppl / 2.5 points and sees 27 of them; 2D: 9), each point's expansion and
    evaluation (its surface points or coefficients), and one far-field translation of each
    box's interaction list (about 60 occupied boxes of 189; 2D: 27), a box per leaf and a
    fifth more."""
    n, nt, method, p = case["n"], case["nt"], case["method"], case["p"]
    if case["kind"] == "served":
        one = [work(_case("", "solve", "cube" if k % 10 in (0, 1, 3, 4, 6, 7, 9) else "yukawa", int(0.47 * n),
                          p=8 if k % 10 in (0, 1, 3, 4, 6, 7, 9) else 10)) for k in range(nt)]
        return {"bytes": sum(w["bytes"] for w in one), "flops": sum(w["flops"] for w in one)}
    nd = {"stokes": 9, "dipole": 4}.get(method, 1)
    nout = {"stokes": 3, "dipole": 4}.get(method, 1)
    dim = 2 if method == "circle" else 3
    leaf = case["ppl"] / 2.5
    boxes = 1.2 * n / leaf
    pair = {"stokes": 55, "dipole": 35, "yukawa": 30, "circle": 25}.get(method, 11)
    if method == "cube":
        coef, trans = (2 * p) ** 3 - (2 * p - 2) ** 3, 60 * 8 * (2 * p - 1) ** 3 // 2
    elif method == "circle":
        coef, trans = p, 27 * 2 * p * p
    else:
        nb = 4 if method == "stokes" else 1
        coef, trans = nb * (p + 1) ** 2, 60 * nb * 2 * (p + 1) ** 3
    src_out = 0 if case["kind"] == "field" else n
    tgt = nt if case["kind"] in ("solve", "field", "circle") else 0
    per = 1.8 if tgt and method == "cube" else 1.0
    flops = pair * (n * coef + (src_out + per * tgt) * (coef + (9 if dim == 2 else 27) * leaf)) + boxes * trans
    byts = 8 * (n * (dim + nd) + src_out * nout + tgt * (dim + (4 if method == "cube" else nout)))
    return {"bytes": float(byts), "flops": float(flops)}


# ---------------------------------------------------------------------------
# the outputs in 64 bits: direct sums
# ---------------------------------------------------------------------------
TB, SB = 512, 32768      # targets and sources per block of a direct sum


def _order(x):
    """A Morton order of points in the unit box (compact blocks of targets)."""
    c = (x * 128).clamp_(0, 127).to(torch.int64)
    key = torch.zeros(x.shape[0], dtype=torch.int64, device=x.device)
    for b in range(7):
        for k in range(3):
            key |= ((c[:, k] >> b) & 1) << (3 * b + k)
    return torch.argsort(key)


def _direct_scalar(x, q, t, kappa=0.0, gradient=False, dipole=False):
    """Potential (and gradient) at t (None: at the sources, each without itself) of
    charges q, kernel exp(-kappa r) / (4 pi r); squared distances as a product of
    coordinates relative to the target block's centre."""
    o = _order(x)
    xs, qs = x[o], q[o]
    to = o if t is None else _order(t)
    ts = xs if t is None else t[to]
    out = torch.empty((ts.shape[0], 4 if gradient else 1), dtype=torch.float64, device=x.device)
    for a in range(0, ts.shape[0], TB):
        b = min(a + TB, ts.shape[0])
        c = ts[a:b].mean(0)
        xi = ts[a:b] - c
        L = torch.cat([xi, (xi * xi).sum(1, keepdim=True), torch.ones_like(xi[:, :1])], 1)
        u = torch.zeros(b - a, dtype=torch.float64, device=x.device)
        g = torch.zeros(b - a, 4, dtype=torch.float64, device=x.device)
        for s0 in range(0, xs.shape[0], SB):
            s1 = min(s0 + SB, xs.shape[0])
            z, qq = xs[s0:s1] - c, qs[s0:s1]
            r2 = L @ torch.cat([-2 * z, torch.ones_like(z[:, :1]), (z * z).sum(1, keepdim=True)], 1).T
            if t is None and s0 <= a < s1:
                r2[:, a - s0:b - s0].diagonal().fill_(math.inf)
            if kappa:
                r = r2.sqrt_()
                w = torch.exp(-kappa * r).div_(r)
                if t is None and s0 <= a < s1:
                    w[:, a - s0:b - s0].diagonal().fill_(0.0)
                u += w @ qq
                continue
            w = r2.rsqrt_()
            u += w @ qq
            if gradient:
                w3 = torch.mul(w, w).mul_(w)
                g += w3 @ torch.cat([qq[:, None], qq[:, None] * z], 1)
        out[to[a:b], 0] = u
        if gradient:
            out[to[a:b], 1:] = g[:, 1:] - xi * g[:, :1]
    out /= 4 * math.pi
    return out if gradient else out[:, 0]


def _blocks(x, t, skip_self, nb):
    """Blocks (targets [a, b), sources [s0, s1), differences d, 1/r with the target itself at 0)."""
    tt = x if t is None else t
    for a in range(0, tt.shape[0], nb):
        b = min(a + nb, tt.shape[0])
        for s0 in range(0, x.shape[0], 8192):
            s1 = min(s0 + 8192, x.shape[0])
            d = [tt[a:b, k, None] - x[None, s0:s1, k] for k in range(3)]
            r2 = d[0] * d[0]
            r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
            lo, hi = max(a, s0), min(b, s1)
            if t is None and lo < hi:
                r2[lo - a:hi - a, lo - s0:hi - s0].diagonal().fill_(math.inf)
            yield a, b, s0, s1, d, r2.rsqrt_()


def _dot(d, v):
    return (d[0] * v[:, 0]).addcmul_(d[1], v[None, :, 1]).addcmul_(d[2], v[None, :, 2])


def _direct_stokes(x, rows, t):
    """The velocity of stokeslets f and stresslets (g, nu), rows [f, g, nu]."""
    tt = x if t is None else t
    u = torch.zeros(tt.shape[0], 3, dtype=torch.float64, device=x.device)
    for a, b, s0, s1, d, w in _blocks(x, t, t is None, 256):
        f, g, nu = rows[s0:s1, 0:3], rows[s0:s1, 3:6], rows[s0:s1, 6:9]
        u[a:b] += w @ f
        w2 = w * w
        w3 = w2 * w
        e = _dot(d, f).addcmul_(_dot(d, g).mul_(_dot(d, nu)), w2, value=-6.0).mul_(w3)
        for k in range(3):
            u[a:b, k] += (e * d[k]).sum(1)
    return u / (8 * math.pi)


def _direct_dipole(x, rows, t):
    """Potential and gradient of charges and dipoles, rows [q, p]."""
    out = torch.zeros(x.shape[0], 4, dtype=torch.float64, device=x.device)
    for a, b, s0, s1, d, w in _blocks(x, t, True, 256):
        q, p = rows[s0:s1, 0], rows[s0:s1, 1:4].contiguous()
        w2 = w * w
        w3 = w2 * w
        pd = _dot(d, p)
        out[a:b, 0] += w @ q + (pd * w3).sum(1)
        e = w3 * q + 3.0 * pd * w3 * w2
        gp = w3 @ p
        for k in range(3):
            out[a:b, 1 + k] += gp[:, k] - (e * d[k]).sum(1)
    return out / (4 * math.pi)


def _direct_circle(x, q, t):
    tt = x if t is None else t
    out = torch.zeros(tt.shape[0], dtype=torch.float64, device=x.device)
    for a in range(0, tt.shape[0], TB):
        b = min(a + TB, tt.shape[0])
        for s0 in range(0, x.shape[0], SB):
            s1 = min(s0 + SB, x.shape[0])
            dx, dy = tt[a:b, 0, None] - x[None, s0:s1, 0], tt[a:b, 1, None] - x[None, s0:s1, 1]
            r2 = dx.mul_(dx).addcmul_(dy, dy)
            lo, hi = max(a, s0), min(b, s1)
            if t is None and lo < hi:
                r2[lo - a:hi - a, lo - s0:hi - s0].diagonal().fill_(1.0)
            out[a:b] += r2.log_() @ q[s0:s1]
    return -out / (4 * math.pi)


def exact(case, seed):
    if case["kind"] == "served":
        put = lambda a: torch.from_numpy(a).to(DEV)   # noqa: E731
        return [_direct_scalar(put(x), put(q), None, 0.0 if lap else KAPPA).cpu().numpy()
                for lap, x, q, _ in _requests(case, seed)]
    x, d, t = _inputs(case, seed)
    method, kind = case["method"], case["kind"]
    if method == "circle":
        return [_direct_circle(x, d, None), _direct_circle(x, d, t)]
    if method == "stokes":
        u = _direct_stokes(x, d, t)
        return u.cpu().numpy() if kind == "stokes_api" else u
    if method == "dipole":
        return _direct_dipole(x, d, None)
    if method == "yukawa":
        return _direct_scalar(x, d, None, KAPPA)
    if kind == "field":
        return _direct_scalar(x, d, t, gradient=True)
    u = _direct_scalar(x, d, None)
    if kind == "host":
        return u.cpu().numpy()
    return u if t is None else [u, _direct_scalar(x, d, t, gradient=True)]
