"""Timed cases: what a program that uses this package has it do.

A case is one pass of a public entry point over a mesh of a stated size: an
LSRK45 step of one problem (one fused launch per stage, or the reference's three
kernels), graph-replayed steps, a step of an ensemble, a forward run with its
discrete adjoint, the diagnostics.  All arithmetic is FP64, the only type the
package has.

    listed()             the cases, smallest calls to the largest
    draw(rng)            another case of the same ranges
    prepare(case, seed)  inputs on the GPU and the solver a program keeps
    run(state)           one pass; returns the whole updated state (see _outputs)
    work(case)           bytes and flops the pass cannot do without
    exact(case, seed)    what run returns on a new state, in plain torch float64

The initial state depends on the seed (2D: strength and centre of the vortex, 3D:
a shift of the Taylor-Green vortex along each axis, or the waves of the varying
state); the mesh depends on the case alone and is kept between preparations.
"""

import dataclasses
import functools
import math
import random

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from scratch_wadge_amd import _lib
from scratch_wadge_amd import mesh as meshes
from scratch_wadge_amd import problem as P
from scratch_wadge_amd import workmodel as W

DEVICE = "cuda:0"

# Share of the default time step: a timed state goes through many thousand
# passes and stays an ordinary flow.
DT_SCALE = {"vortex": 0.25, "tgv": 0.5, "varying": 0.02}


def listed():
    return [
        # the smallest 2D run: one eager step, five launches, latency only
        dict(name="vortex2d_N2_K128_step", kind="step", dim=2, N=2, n=8, curved=False,
             state="vortex", fused=True),
        # an ordinary 2D run stepped from a HIP graph (the adjoint's forward uses it too)
        dict(name="vortex2d_N3_K2048_graph", kind="graph", dim=2, N=3, n=32, curved=False,
             state="vortex", steps=4),
        # a large 2D run; 2 * 127^2 elements fill no launch shape evenly
        dict(name="vortex2d_N4_K32258_step", kind="step", dim=2, N=4, n=127, curved=False,
             state="vortex", fused=True),
        # a small 3D run on curved tets: a coarse mesh of a convergence study
        dict(name="tgv3d_N3_K2058_step", kind="step", dim=3, N=3, n=7, curved=True, state="tgv",
             fused=True),
        # the reference's three kernels per stage on affine tets, 16^3 x 6
        dict(name="tgv3d_N3_K24576_split", kind="step", dim=3, N=3, n=16, curved=False,
             state="tgv", fused=False),
        # the headline workload: curved Taylor-Green, 32^3 x 6
        dict(name="tgv3d_N3_K196608_step", kind="step", dim=3, N=3, n=32, curved=True, state="tgv",
             fused=True),
        # high order on curved tets, an odd element count per cube edge
        dict(name="tgv3d_N4_K13182_step", kind="step", dim=3, N=4, n=13, curved=True, state="tgv",
             fused=True),
        # low order, a strongly varying state: both branches of the log mean
        dict(name="varying3d_N2_K48000_step", kind="step", dim=3, N=2, n=20, curved=True,
             state="varying", fused=True),
        # 64 independent 2D problems of uneven K and N in one launch per stage
        dict(name="ensemble2d_64_graph", kind="ensemble", count=64, kmin=128, kmax=8192, steps=2,
             draw_seed=0),
        # forward run and adjoint sweep of a 2D problem, recomputed from checkpoints
        dict(name="adjoint2d_N3_K2048", kind="adjoint", dim=2, N=3, n=32, curved=False,
             state="vortex", steps=8, every=4),
        # the same on curved tets
        dict(name="adjoint3d_N3_K10368", kind="adjoint", dim=3, N=3, n=12, curved=True, state="tgv",
             steps=2, every=1),
        # energy, entropy, mass and error of a run, as printed every few steps
        dict(name="diagnostics3d_N3_K82944", kind="diagnostics", dim=3, N=3, n=24, curved=True,
             state="varying"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["step", "step", "step", "graph", "ensemble", "adjoint", "adjoint",
                       "diagnostics"])
    if kind == "ensemble":
        kmin = _log_int(rng, 32, 256)
        return dict(kind=kind, count=rng.randint(4, 48), kmin=kmin,
                    kmax=kmin * rng.randint(2, 24), steps=rng.randint(1, 3),
                    draw_seed=rng.randrange(1 << 20))
    dim = rng.choice([2, 3])
    N = rng.randint(1, 5) if dim == 2 else rng.randint(1, 4)
    c = dict(kind=kind, dim=dim, N=N)
    small = kind == "adjoint"
    if dim == 2:
        c["n"] = _log_int(rng, 4, 64 if small else 160)
        c["curved"] = False
        c["state"] = rng.choice(["vortex", "vortex", "varying"])
    else:
        c["n"] = _log_int(rng, 3, (12 if N < 4 else 8) if small else (22 if N < 4 else 14))
        c["curved"] = rng.random() < 0.6
        c["state"] = rng.choice(["tgv", "tgv", "varying"])
    if kind == "step":
        c["fused"] = rng.random() < 0.7
    elif kind == "graph":
        c["steps"] = 2 * rng.randint(1, 3)
    elif kind == "adjoint":
        c["state"] = "vortex" if dim == 2 else "tgv"
        c["steps"] = rng.randint(1, 3) if dim == 3 else rng.randint(2, 8)
        c["every"] = rng.randint(1, 4)
    elif dim == 3:
        c["state"] = "varying"        # a shifted Taylor-Green vortex has the same totals
    return c


def _outputs(case):
    """The state a step leaves behind.  resQ, the register of the RK stages, is
    dead after a whole step (the first stage's coefficient is zero).  It is
    returned for the varying state; in the vortex and the Taylor-Green vortex it
    is the small remainder of fluxes that cancel, whose digits follow the
    round-off of the state (one unit in the last place of Q moves it by 1e-10 to
    1e-8 of its norm)."""
    names = ("Q", "rhsQ", "Qf")
    return names + ("resQ",) if case.get("state") == "varying" else names


# ------------------------------------------------------------------ inputs

@functools.lru_cache(maxsize=3)
def _base(dim, N, n, curved):
    """Mesh, geometry and operators of a case (host arrays)."""
    if dim == 2:
        return P.vortex2d_problem(n=n, N=N)
    return P.tgv3d_problem(n=n, N=N, curved=curved)


def _problem(case, seed):
    base = _base(case["dim"], case["N"], case["n"], case["curved"])
    rng = np.random.default_rng(seed)
    if case["state"] == "varying":
        # on the coarsest meshes the face extrapolation of strong waves leaves
        # the admissible set
        amp = 0.2 if case["dim"] == 2 and case["n"] >= 8 else 0.08 if case["n"] >= 6 else 0.03
        Q, uq, uf = P.varying_state(base, seed=seed, amp=amp)
    else:
        if case["dim"] == 2:
            U = P.vortex_2d(*base.xq, 0.0, *rng.uniform(-2, 2, size=2),
                            beta=rng.uniform(1, 3))
        else:
            s = rng.uniform(0, 2 * np.pi, size=3)
            U = P.taylor_green(*(x + d for x, d in zip(base.xq, s)))
        Q, uq, uf = (np.ascontiguousarray(a.transpose(2, 0, 1)).reshape(-1)
                     for a in P.project_initial_state(base.ops, U, base.gamma))
    return dataclasses.replace(base, Q=Q, rhsQ=uq, Qf=uf, resQ=np.zeros_like(Q),
                               dt=base.dt * DT_SCALE[case["state"]])


def _adjoint_inputs(case, prob, seed):
    """Initial state with one part in a thousand of scatter (measured data), and
    the target of a squared misfit."""
    rng = np.random.default_rng(seed + 1)
    Q0 = prob.Q * (1.0 + 1e-3 * rng.standard_normal(prob.Q.shape))
    target = prob.Q * (1.0 + 1e-2 * rng.standard_normal(prob.Q.shape))
    return Q0, target


def _ensemble_problems(case, seed):
    """Meshes and degrees from the case, vortices from the seed."""
    rng = np.random.default_rng(case["draw_seed"])
    vort = np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        k = math.exp(rng.uniform(math.log(case["kmin"]), math.log(case["kmax"])))
        n = max(4, int(round(math.sqrt(k / 2.0))))
        N = int(rng.choice((2, 3, 4)))
        x0, y0 = vort.uniform(-2, 2, size=2)
        out.append(P.vortex2d_problem(n=n, N=N, beta=float(vort.uniform(1, 3)), x0=float(x0),
                                      y0=float(y0), seed=n))
    return [dataclasses.replace(p, dt=p.dt * DT_SCALE["vortex"]) for p in out]


def _slots(sizes):
    """Offsets of arrays in one flat buffer, 64 doubles aligned, and its length."""
    off, at = [], 0
    for s in sizes:
        off.append(at)
        at += -(-s // 64) * 64
    return off, at


def prepare(case, seed):
    from scratch_wadge_amd.adjoint import AdjointSolver
    from scratch_wadge_amd.device import DeviceSolver
    from scratch_wadge_amd.ensemble import group_of
    kind = case["kind"]
    if kind == "ensemble":
        probs = _ensemble_problems(case, seed)
        solvers = [DeviceSolver(p, DEVICE) for p in probs]
        flat = {}
        for name in ("Q", "rhsQ", "resQ", "Qf", "Qf_alt"):
            own = [sv.Qf_alt if name == "Qf_alt" else sv.s[name] for sv in solvers]
            off, length = _slots([t.numel() for t in own])
            flat[name] = torch.zeros(length, dtype=torch.float64, device=DEVICE)
            for sv, t, o in zip(solvers, own, off):
                view = flat[name][o:o + t.numel()]
                view.copy_(t)
                if name == "Qf_alt":
                    sv.Qf_alt = view
                else:
                    sv.s[name] = view
        batch = _lib.Batch(2, [group_of(sv) for sv in solvers], probs[0].gamma, probs[0].tau,
                           solvers[0].stream())
        return dict(case=case, batch=batch, solvers=solvers, flat=flat)
    prob = _problem(case, seed)
    dev = DeviceSolver(prob, DEVICE)
    st = dict(case=case, dev=dev, dt=prob.dt)
    if kind == "adjoint":
        Q0, target = _adjoint_inputs(case, prob, seed)
        st["Q0"] = torch.as_tensor(Q0, device=DEVICE)
        st["target"] = torch.as_tensor(target, device=DEVICE)
        st["adj"] = AdjointSolver(dev, checkpoint_every=case["every"])
    elif kind == "diagnostics":
        st["exact_state"] = torch.as_tensor(prob.Q * (1.0 + 1e-3), device=DEVICE)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "ensemble":
        b, f = st["batch"], st["flat"]
        b.run(case["steps"], True, st["solvers"][0].stream())
        return {"Q": f["Q"], "rhsQ": f["rhsQ"], "Qf": f["Qf"] if b.current() == 0 else f["Qf_alt"]}
    dev = st["dev"]
    if kind == "diagnostics":
        return dev.diagnostics(st["exact_state"])
    if kind == "adjoint":
        adj = st["adj"]
        QT = adj.forward(st["Q0"], case["steps"], st["dt"])
        return {"QT": QT, "grad": adj.backward(QT - st["target"])}
    if kind == "graph":
        dev.run(case["steps"], st["dt"], fused=True, graph=True)
    else:
        dev.step(st["dt"], fused=case["fused"])
    return {k: dev.s[k] for k in _outputs(case)}


# ------------------------------------------------------------------ work

def _stage_work(dim, Nq, Nf):
    return W.bytes_stage_fused(dim, Nq, Nf), W.stage_flops(dim, Nq, Nf)


@functools.lru_cache(maxsize=None)
def _shape(dim, N):
    from scratch_wadge_amd.operators import build_ref_ops
    o = build_ref_ops(dim, N)
    return o.Nq, o.Nf


def work(case):
    if case["kind"] == "ensemble":
        rng = np.random.default_rng(case["draw_seed"])
        b = f = 0.0
        for _ in range(case["count"]):
            k = math.exp(rng.uniform(math.log(case["kmin"]), math.log(case["kmax"])))
            n = max(4, int(round(math.sqrt(k / 2.0))))
            sb, sf = _stage_work(2, *_shape(2, int(rng.choice((2, 3, 4)))))
            b += 2 * n * n * sb
            f += 2 * n * n * sf
        return {"bytes": 5 * case["steps"] * b, "flops": 5 * case["steps"] * f}
    dim = case["dim"]
    Nq, Nf = _shape(dim, case["N"])
    K = 2 * case["n"] ** 2 if dim == 2 else 6 * case["n"] ** 3
    sb, sf = _stage_work(dim, Nq, Nf)
    if case["kind"] == "diagnostics":
        # Q, the exact state and J in
        return {"bytes": 8.0 * K * Nq * (2 * (dim + 2) + 1), "flops": K * Nq * (8.0 * dim + 20)}
    if case["kind"] == "adjoint":
        # forward stages, recomputed stages of all segments but the last, and
        # reverse stages; a reverse stage reads the recorded states and the
        # cotangents, and differentiates every flux and map of a stage (counted
        # as twice the stage's flops)
        n, c = case["steps"], case["every"]
        again = (n - 1) // c * c
        nf = dim + 2
        rb = 8 * (nf * (Nq + 2 * Nf) + dim * dim * (Nq + Nf) + 2 * (dim + 1) * Nf + Nq
                  + nf * (7 * Nq + 4 * Nf)) + 4 * Nf
        return {"bytes": 5.0 * K * ((n + again) * sb + n * rb),
                "flops": 5.0 * K * (n + again + 2 * n) * sf}
    steps = case.get("steps", 1)
    if not case.get("fused", True):
        # the three kernels are separate calls: what each of them reads and writes
        sb = W.bytes_vol(dim, Nq, Nf) + W.bytes_surf(dim, Nq, Nf) + W.bytes_update(dim, Nq, Nf)
    return {"bytes": 5.0 * steps * K * sb, "flops": 5.0 * steps * K * sf}


# ------------------------------------------------------------------ plain float64 values

class _Ops:
    def __init__(self, prob):
        dev = DEVICE if torch.cuda.is_available() else "cpu"
        T = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=dev)
        o = prob.ops
        dim, K, Nq, Nf = prob.dim, prob.K, prob.Nq, prob.Nf
        self.dim, self.K, self.Nq, self.Nf, self.nf = dim, K, Nq, Nf, dim + 2
        self.gamma, self.tau, self.dt = prob.gamma, prob.tau, prob.dt
        self.D = torch.stack([T(d) for d in o.Drst], -1)                      # (Nq, Nq, r)
        self.VqLq, self.VqPq, self.VfPq = T(o.VqLq), T(o.VqPq), T(o.VfPq)
        self.nref = T(o.nref)                                                 # (Nf, r)
        self.vg = T(prob.vgeo).reshape(K, dim, dim, Nq).permute(0, 3, 1, 2)   # (K, Nq, r, d)
        self.fg = T(prob.vfgeo).reshape(K, dim, dim, Nf).permute(0, 3, 1, 2)
        g = T(prob.fgeo).reshape(K, dim + 1, Nf)
        self.nJ, self.sJ = g[:, :dim].permute(0, 2, 1), g[:, dim]
        self.nbr = torch.as_tensor(prob.mapPq.astype(np.int64), device=dev).reshape(K, Nf)
        self.J = T(prob.Jq).reshape(K, 1, Nq)
        self.T = T


def _logmean(a, b):
    """(a - b) / (ln a - ln b), accurate for a near b."""
    d = a - b
    f = d / (a + b)
    u = f * f
    near = u < 1e-3
    ser = 0.5 * (a + b) / (1 + u * (1 / 3 + u * (1 / 5 + u * (1 / 7 + u * (1 / 9 + u / 11)))))
    ds = torch.where(near, torch.ones_like(d), d)
    bs = torch.where(near, torch.ones_like(b), b)
    return torch.where(near, ser, ds / torch.log1p(ds / bs))


def _prim(U, g):
    """(..., nf) -> rho, velocity, beta, p, |u|^2."""
    rho = U[..., 0]
    vel = U[..., 1:-1] / rho[..., None]
    uu = (vel * vel).sum(-1)
    p = (g - 1.0) * (U[..., -1] - 0.5 * rho * uu)
    return rho, vel, rho / (2.0 * p), p, uu


def _flux(A, B, n, g):
    """Entropy-conservative two-point flux along n (..., d): (..., nf)."""
    rl, bl = _logmean(A[0], B[0]), _logmean(A[2], B[2])
    va = 0.5 * (A[1] + B[1])
    vn = 2.0 * (va * va).sum(-1) - 0.5 * (A[4] + B[4])
    pa = 0.5 * (A[0] + B[0]) / (A[2] + B[2])
    Un = (va * n).sum(-1)
    m = rl * Un
    e = (rl / (2.0 * (g - 1.0) * bl) + pa + 0.5 * rl * vn) * Un
    return torch.cat([m[..., None], m[..., None] * va + pa[..., None] * n, e[..., None]], -1)


def _vol_chunk(o, uq, uf, vg, fg):
    """Volume rows and face rows of some elements; uq (k, Nq, nf), uf (k, Nf, nf)."""
    q, f = _prim(uq, o.gamma), _prim(uf, o.gamma)
    row = tuple(x[:, :, None] for x in q)
    n = torch.einsum("ijr,kird->kijd", 0.5 * o.D, vg) + torch.einsum("ijr,kjrd->kijd", 0.5 * o.D, vg)
    r = _flux(row, tuple(x[:, None] for x in q), n, o.gamma).sum(2)
    n = 0.5 * (torch.einsum("jr,kird->kijd", o.nref, vg)
               + torch.einsum("jr,kjrd->kjd", o.nref, fg)[:, None])
    F = _flux(row, tuple(x[:, None] for x in f), n, o.gamma)
    r = r + 0.5 * (o.VqLq[None, :, :, None] * F).sum(2)
    return r, -0.5 * (o.VfPq.T[None, :, :, None] * F).sum(1)


def _rhs(o, uq, uf):
    """RHS (K, nf, Nq) of projected states uq (K, nf, Nq), uf (K, nf, Nf)."""
    uqT, ufT = uq.transpose(1, 2), uf.transpose(1, 2)
    step = max(1, int(1_500_000 // (o.Nq * (o.Nq + o.Nf))))
    parts = [checkpoint(_vol_chunk, o, uqT[k:k + step], ufT[k:k + step], o.vg[k:k + step],
                        o.fg[k:k + step], use_reentrant=False) if uq.requires_grad else
             _vol_chunk(o, uqT[k:k + step], ufT[k:k + step], o.vg[k:k + step], o.fg[k:k + step])
             for k in range(0, o.K, step)]
    r = torch.cat([x[0] for x in parts])
    rf = torch.cat([x[1] for x in parts])
    idx = o.nbr[:, :, None] + o.Nf * torch.arange(o.nf, device=uf.device)
    UP = uf.reshape(-1)[idx]
    M, Pp = _prim(ufT, o.gamma), _prim(UP, o.gamma)
    lam = torch.maximum(torch.sqrt(M[4]) + torch.sqrt(o.gamma * M[3] / M[0]),
                        torch.sqrt(Pp[4]) + torch.sqrt(o.gamma * Pp[3] / Pp[0]))
    s = (0.5 * _flux(M, Pp, o.nJ, o.gamma) + rf
         - (0.25 * o.tau * lam * o.sJ)[..., None] * (UP - ufT))
    return (r + torch.einsum("ij,kjf->kif", o.VqLq, s)).transpose(1, 2)


def _entropy(U, g):
    """(..., nf) -> entropy variables."""
    rho, E = U[..., 0], U[..., -1]
    rhoe = E - 0.5 * (U[..., 1:-1] ** 2).sum(-1) / rho
    s = torch.log((g - 1.0) * rhoe) - g * torch.log(rho)
    return torch.cat([(g + 1.0 - s - E / rhoe)[..., None], U[..., 1:-1] / rhoe[..., None],
                      (-rho / rhoe)[..., None]], -1)


def _conservative(V, g):
    vl = V[..., -1]
    h = (V[..., 1:-1] ** 2).sum(-1) / (2.0 * vl)
    rhoe = torch.exp((math.log(g - 1.0) - g * torch.log(-vl) - (g - V[..., 0] + h)) / (g - 1.0))
    return torch.cat([(-rhoe * vl)[..., None], rhoe[..., None] * V[..., 1:-1],
                      (rhoe * (1.0 - h))[..., None]], -1)


def _project(o, vt):
    """u(v~) and u(VfPq v~) of entropy variables vt (K, Nq, nf)."""
    return (_conservative(vt, o.gamma).transpose(1, 2),
            _conservative(torch.einsum("ij,kjf->kif", o.VfPq, vt), o.gamma).transpose(1, 2))


def _step(o, Q, res, uq, uf, dt):
    for a, b in zip(P.RK4A, P.RK4B):
        R = _rhs(o, uq, uf)
        r = torch.einsum("ij,kfj->kfi", -2.0 * o.VqPq, R) / o.J
        res = a * res + dt * torch.einsum("ij,kfj->kfi", o.VqPq, r)
        Q = Q + b * res
        V = _entropy(Q.transpose(1, 2), o.gamma) * o.J.transpose(1, 2)
        w = torch.einsum("ij,kjf->kif", o.VqPq, V) / o.J.transpose(1, 2)
        uq, uf = _project(o, torch.einsum("ij,kjf->kif", o.VqPq, w))
    return Q, res, uq, uf


def _steps(prob, steps, names):
    o = _Ops(prob)
    sh = lambda a, n: o.T(a).reshape(o.K, o.nf, n)
    s = (sh(prob.Q, o.Nq), sh(prob.resQ, o.Nq), sh(prob.rhsQ, o.Nq), sh(prob.Qf, o.Nf))
    for _ in range(steps):
        s = _step(o, *s, o.dt)
    s = dict(zip(("Q", "resQ", "rhsQ", "Qf"), s))
    return {k: s[k].contiguous().reshape(-1) for k in names}


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        parts = [_steps(p, case["steps"], _outputs(case)) for p in _ensemble_problems(case, seed)]
        out = {}
        for name in _outputs(case):
            off, length = _slots([p[name].numel() for p in parts])
            out[name] = torch.zeros(length, dtype=torch.float64, device=parts[0][name].device)
            for p, o in zip(parts, off):
                out[name][o:o + p[name].numel()] = p[name]
        return out
    prob = _problem(case, seed)
    if kind == "diagnostics":
        o = _Ops(prob)
        U = o.T(prob.Q).reshape(o.K, o.nf, o.Nq)
        wJ = o.T(prob.wq) * o.J[:, 0]
        mm = (U[:, 1:-1] ** 2).sum(1)
        s = torch.log((o.gamma - 1.0) * (U[:, -1] - 0.5 * mm / U[:, 0])) - o.gamma * torch.log(U[:, 0])
        err = ((U - U * (1.0 + 1e-3)) ** 2).sum(1)
        return {"kinetic_energy": float((0.5 * wJ * mm / U[:, 0]).sum()),
                "entropy": float((-wJ * U[:, 0] * s).sum()),
                "l2_error": float((wJ * err).sum()) ** 0.5, "mass": float((wJ * U[:, 0]).sum())}
    if kind == "adjoint":
        o = _Ops(prob)
        Q0, target = (o.T(a).reshape(o.K, o.nf, o.Nq) for a in _adjoint_inputs(case, prob, seed))
        Q0.requires_grad_(True)
        V = _entropy(Q0.transpose(1, 2), o.gamma)
        # the initial projection: u(VqPq v), u(VfPq v)
        uq, uf = (_conservative(torch.einsum("ij,kjf->kif", A, V), o.gamma).transpose(1, 2)
                  for A in (o.VqPq, o.VfPq))
        s = (Q0, torch.zeros_like(Q0), uq, uf)
        for _ in range(case["steps"]):
            s = _step(o, *s, o.dt)
        QT = s[0]
        (g,) = torch.autograd.grad(QT, Q0, (QT - target).detach())
        return {"QT": QT.detach().contiguous().reshape(-1), "grad": g.contiguous().reshape(-1)}
    return _steps(prob, case.get("steps", 1), _outputs(case))
