#!/usr/bin/env python3
"""Benchmark of the WADGES RK stage on one MI355X.

Workload (default): 3D Taylor-Green vortex on the warped periodic cube,
32^3 cubes x 6 tetrahedra (K = 196,608), N = 3 (Np = 20, Nq = 23, Nf = 48),
FP64, tau = 1.  A step is one LSRK45 time step = 5 stages of
vol -> surf -> update over all elements, with every array resident in HBM.

Metric: GDOF.RK-stage/s = K * Np * Nfields * stages / time / 1e9.
The timed region runs the fused stage kernel (one launch per stage); the
three-kernel path (vol -> surf -> update, the reference's structure) is timed
beforehand for the per-kernel breakdown.  Prints one JSON line.  The roofline
object is for the fused stage kernel: achieved = algorithmic FP64 flops per
launch (workmodel: volume with each flux counted once, plus surface and
update) / mean launch time measured with HIP events on the launch stream.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--n", type=int, default=32, help="cubes per direction")
    ap.add_argument("--N", type=int, default=3, help="polynomial degree")
    ap.add_argument("--affine", action="store_true")
    ap.add_argument("--cpu-baseline", dest="cpu", action="store_true", default=True)
    ap.add_argument("--no-cpu-baseline", dest="cpu", action="store_false")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--extras", dest="extras", action="store_true", default=True,
                    help="also measure the ensemble and adjoint workloads (default)")
    ap.add_argument("--no-extras", dest="extras", action="store_false")
    ap.add_argument("--ensemble-steps", type=int, default=100)
    ap.add_argument("--leg", choices=("all", "ensemble", "adjoint", "adjoint3d"), default="all",
                    help="ensemble / adjoint: run only that leg and print its JSON object; "
                         "adjoint3d: the adjoint sweep on the 3D curved K = 196,608, N = 3 mesh "
                         "(not part of the default run)")
    ap.add_argument("--adjoint-steps", type=int, default=400)
    ap.add_argument("--copy-calibration", type=float, default=0.0, metavar="GIB",
                    help="instead of the benchmark, copy a GIB-sized device buffer 5 times "
                         "(reference kernel of known traffic for the HBM counters)")
    return ap.parse_args()


def copy_calibration(gib):
    import torch
    n = int(gib * (1 << 30)) // 8
    a = torch.ones(n, dtype=torch.float64, device="cuda:0")
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    for _ in range(5):
        b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration": {"bytes_read_per_copy": n * 8,
                                            "bytes_written_per_copy": n * 8, "copies": 5}}))


def cpu_baseline(prob, target_s):
    """The CPU oracle (OpenMP over elements) timed on the host cores on a sample
    of elements of the same workload; returns GDOF.stage/s."""
    import numpy as np
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import pyoracle as O
    O.build()
    threads = min(16, os.cpu_count() or 1)
    O.set_threads(threads)
    st = {k: v.copy() for k, v in prob.copy_state().items()}
    rf = np.zeros_like(st["Qf"])
    par = O.params(prob)
    L = O.lib()
    import ctypes

    def stage(Ks):
        p = O._p
        L.wo_vol(ctypes.byref(par), Ks, p(prob.vgeo), p(prob.vfgeo), p(prob.nrJ), p(prob.nsJ),
                 p(prob.ntJ), p(prob.Drq), p(prob.Dsq), p(prob.Dtq), p(prob.VqLq), p(prob.VfPq),
                 p(st["Qf"]), p(st["rhsQ"]), p(rf))
        m = np.ascontiguousarray(prob.mapPq, dtype=np.uint32)
        L.wo_surf(ctypes.byref(par), Ks, p(prob.fgeo), m.ctypes.data_as(O._up), p(prob.VqLq),
                  p(st["Qf"]), p(rf), p(st["rhsQ"]))
        L.wo_update(ctypes.byref(par), Ks, p(prob.Jq), p(prob.VqPq), p(prob.VfPq), 0.0, 0.1,
                    1e-4, p(st["rhsQ"]), p(st["resQ"]), p(st["Q"]), p(st["Qf"]))

    Ks = min(prob.K, 256 * threads)
    t0 = time.perf_counter()
    stage(Ks)
    t1 = time.perf_counter() - t0
    Ks = int(min(prob.K, max(Ks, Ks * target_s / max(t1, 1e-6))))
    Ks -= Ks % threads if Ks > threads else 0
    # whole stages over Ks elements until about target_s of work (at most 50)
    reps, dt = 0, 0.0
    t0 = time.perf_counter()
    while reps < 50 and (reps == 0 or dt < target_s):
        stage(Ks)
        reps += 1
        dt = time.perf_counter() - t0
    from scratch_wadge_amd.workmodel import dofs
    gdof = dofs(prob.dim, prob.N, Ks) * reps / dt / 1e9
    return {"value": gdof, "unit": "GDOF*stage/s", "cores": threads, "kind": "port",
            "sample": f"{reps} vol+surf+update stages over {Ks} of {prob.K} elements "
                      f"({dt:.1f} s, C++ oracle, OpenMP {threads} threads)"}


def profiled_value(key, kernel, workload_file):
    """A per-launch figure of `kernel` recorded in a committed rocprofv3 summary
    under profiles/ (lines "key kernel value"), or None when no summary covers
    this workload.  Keys: traffic_bytes_per_launch (FETCH_SIZE / WRITE_SIZE
    passes scaled by the copy-kernel calibration), fp64_lane_flops_per_launch
    (64 (ADD + MUL + TRANS) + 128 FMA from the SQ_INSTS_VALU_*_F64 pass),
    kernel_avg_us (the kernel-trace average)."""
    path = os.path.join(ROOT, "profiles", workload_file)
    if not os.path.exists(path):
        return None
    for line in open(path):
        parts = line.split()
        if len(parts) == 3 and parts[0] == key and parts[1] == kernel:
            return float(parts[2])
    return None


def _sync_time(fn):
    import torch
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    fn()
    torch.cuda.synchronize()
    return time.perf_counter() - t0


def ensemble_bench(steps, seed=0):
    """64 independent 2D vortex problems (K log-uniform in [128, 8192], N in
    {2,3,4}, strength U[3,6], centre U[-2,2]^2): the ensemble kernel with its
    graph-replayed step against one wadges_stage launch per problem per stage."""
    import numpy as np
    from scratch_wadge_amd.ensemble import Ensemble, PerProblem, vortex_ensemble
    t0 = time.perf_counter()
    probs = vortex_ensemble(64, seed=seed)
    ens, base, base_g = Ensemble(probs), PerProblem(probs), PerProblem(probs)
    print(f"# ensemble setup {time.perf_counter() - t0:.1f}s K_total={ens.K_total}",
          file=sys.stderr, flush=True)
    tuned_ms = ens.tune(reps=5)
    t_batch = _sync_time(lambda: ens.run(steps, use_graph=True))
    t_base = _sync_time(lambda: base.run(steps))
    equal = all(np.array_equal(ens.state(q)[f], base.state(q)[f]) for q in range(len(probs))
                for f in ("Q", "rhsQ", "resQ", "Qf"))
    finite = all(np.isfinite(ens.state(q)["Q"]).all() for q in range(len(probs)))
    t_batch_eager = _sync_time(lambda: ens.run(steps, use_graph=False))
    base_g.run(2, use_graph=True)                 # capture outside the timing
    t_base_g = _sync_time(lambda: base_g.run(steps, use_graph=True))
    work = ens.dofs * 5 * steps / 1e9
    # roofline of the ensemble kernel: one launch per stage over all problems
    import torch
    from scratch_wadge_amd import workmodel as W
    stream = torch.cuda.current_stream()
    evs = []
    for _ in range(4):
        for s in range(5):
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record(stream)
            ens.stage(s)
            b.record(stream)
            evs.append((a, b))
    torch.cuda.synchronize()
    launch_ms = float(np.mean([a.elapsed_time(b) for a, b in evs]))
    flops = sum(p.K * W.stage_flops(2, p.Nq, p.Nf) for p in probs)
    achieved = flops / (launch_ms * 1e-3) / 1e12
    g = lambda t: round(work / t, 4)
    return {"workload": "64 2D isentropic vortex problems, K log-uniform in [128, 8192] "
                        "(nearest 2n^2), N in {2,3,4}, strength U[3,6], centre U[-2,2]^2, seed 0",
            "K_total": ens.K_total, "steps": steps, "unit": "GDOF*stage/s",
            "batched_graph": g(t_batch), "batched_eager": g(t_batch_eager),
            "per_problem_eager": g(t_base), "per_problem_graph": g(t_base_g),
            "speedup_vs_per_problem_eager": round(t_base / t_batch, 3),
            "speedup_vs_per_problem_graph": round(t_base_g / t_batch, 3),
            "launch_shape": ens.config(), "tuned_stage_ms": round(tuned_ms, 4),
            "bitwise_equal_to_per_problem": bool(equal), "finite": bool(finite),
            "roofline": {"bound": "fp64 valu", "kernel": "batch_stage_flat",
                         "achieved": round(achieved, 3), "peak": W.FP64_PEAK_TFLOPS,
                         "unit": "TFLOP/s", "frac": round(achieved / W.FP64_PEAK_TFLOPS, 4),
                         "flops_per_launch": flops, "launch_ms": round(launch_ms, 4)}}


def adjoint3d_bench(steps=8, ckpt=4, n=32):
    """The adjoint sweep at the headline scale: 3D curved Taylor-Green, n^3 x 6
    tets (K = 196,608 at n = 32), N = 3, `steps` LSRK45 steps with checkpoints
    every `ckpt`, cotangent of all ones at the final state; sweep time against
    the plain forward (both replayed from HIP graphs)."""
    import torch
    from scratch_wadge_amd import problem as P
    from scratch_wadge_amd.adjoint import AdjointSolver
    from scratch_wadge_amd.device import DeviceSolver
    prob = P.tgv3d_problem(n=n, N=3, curved=True)
    dev = DeviceSolver(prob)
    dev.run(2, fused=True, graph=True)              # warm-up, graph capture
    t_plain = _sync_time(lambda: dev.run(steps, fused=True, graph=True))
    adj = AdjointSolver(dev, checkpoint_every=ckpt)
    Q0 = torch.as_tensor(prob.Q, device=dev.device)
    adj.forward(Q0, steps)                          # warm-up, graph captures
    adj.backward(torch.zeros_like(Q0))
    out = {}
    t_fwd = _sync_time(lambda: out.setdefault("QT", adj.forward(Q0, steps)))
    t_bwd = _sync_time(lambda: out.setdefault("g", adj.backward(torch.ones_like(Q0))))
    g = out["g"]
    kernels = vjp_kernel_times(dev, adj)
    return {"workload": f"3D curved TGV {n}^3 x 6 (K={prob.K}), N=3, {steps} steps, "
                        f"checkpoints every {ckpt}",
            "forward_ms": round(t_plain * 1e3, 2), "forward_with_checkpoints_ms": round(t_fwd * 1e3, 2),
            "adjoint_sweep_ms": round(t_bwd * 1e3, 2),
            "adjoint_over_forward": round(t_bwd / t_plain, 3),
            "grad_finite": bool(torch.isfinite(g).all()), "grad_norm": float(torch.linalg.norm(g)),
            "vjp_kernels": kernels}


def vjp_kernel_times(dev, adj, reps=5):
    """Launch times (HIP events on the launch stream) of the reverse pass's kernels on
    the states the sweep left in its slots: the recorded forward stage, the update
    VJP and the RHS VJP; with the executed FP64 vector-ALU flops per launch of the
    committed rocprofv3 summary (SQ_INSTS_VALU_*_F64) where it covers them, as the
    VJP kernels' roofline (they have no algorithmic count of their own)."""
    import numpy as np
    import torch
    from scratch_wadge_amd import workmodel as W
    from scratch_wadge_amd.device import _ptr
    from scratch_wadge_amd.problem import RK4A, RK4B
    c, K, st = dev.c, dev.K, torch.cuda.current_stream()
    S = adj._ensure_slots()
    P = lambda n: _ptr(c[n])
    geo = (P("vgeo"), P("vfgeo"), P("fgeo"), P("mapPq"), P("nrJ"), P("nsJ"), P("ntJ"), P("Drq"),
           P("Dsq"), P("Dtq"), P("VqLq"), P("VqPq"), P("VfPq"), P("Jq"))
    dt = adj.dt
    res = torch.empty_like(dev.s["Q"])
    Qb, rb = torch.empty_like(dev.s["Q"]), torch.empty_like(dev.s["Q"])
    uqb, ufb = torch.empty_like(dev.s["rhsQ"]), torch.empty_like(dev.s["Qf"])
    rhsb, sbar = torch.empty_like(dev.s["Q"]), torch.empty_like(dev.s["Qf"])
    calls = {
        "stage_record": lambda: dev.plan.stage_record(
            K, *geo, RK4A[1], RK4B[1], dt, _ptr(S["Qf"][0]), _ptr(S["Qf"][1]), _ptr(S["rhsQ"][0]),
            _ptr(S["rhsQ"][1]), _ptr(res), _ptr(res), _ptr(S["Q"][0]), _ptr(S["Q"][1]), st.cuda_stream),
        "update_vjp": lambda: dev.plan.update_vjp(
            K, P("Jq"), P("VqPq"), P("VfPq"), RK4A[1], RK4B[1], dt, _ptr(S["Q"][1]), _ptr(Qb), _ptr(rb),
            _ptr(uqb), _ptr(ufb), _ptr(rhsb), st.cuda_stream),
        "rhs_vjp": lambda: dev.plan.rhs_vjp(
            K, *geo[:11], P("VfPq"), _ptr(S["rhsQ"][0]), _ptr(S["Qf"][0]), _ptr(rhsb), _ptr(sbar),
            _ptr(uqb), _ptr(ufb), st.cuda_stream),
    }
    for t in (Qb, rb, uqb, ufb):
        t.fill_(1e-3)
    out = {}
    prof = lambda key, kernel: profiled_value(key, kernel, "adjoint_sweep_tgv3d_curved_K196608_N3.md")
    for name, fn in calls.items():
        fn()
        evs = []
        for _ in range(reps):
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record(st)
            fn()
            b.record(st)
            evs.append((a, b))
        torch.cuda.synchronize()
        ms = float(np.mean([a.elapsed_time(b) for a, b in evs]))
        entry = {"launch_ms": round(ms, 4)}
        kern = {"stage_record": "team_stage_kernel", "update_vjp": "update_vjp_mfma_kernel",
                "rhs_vjp": "rhs_vjp_kernel"}[name]
        fl = prof("fp64_lane_flops_per_launch", kern)
        if fl is not None:
            tf = fl / (ms * 1e-3) / 1e12
            entry["roofline"] = {"bound": "fp64 valu", "kernel": kern,
                                 "counter_tflops": round(tf, 3), "peak": W.FP64_PEAK_TFLOPS,
                                 "frac": round(tf / W.FP64_PEAK_TFLOPS, 4),
                                 "flops": "executed FP64 vector-ALU lane flops per launch, "
                                          "64 (ADD+MUL+TRANS) + 128 FMA (SQ_INSTS_VALU_*_F64)"}
        out[name] = entry
    return out


def adjoint_bench(steps, ckpt=40):
    """2D vortex, 32x32x2 = 2048 triangles, N=3: density misfit after `steps`
    LSRK45 steps against a target from Gaussian-bump-perturbed initial density;
    times the checkpointed adjoint sweep against the plain forward (both
    replayed from HIP graphs)."""
    import torch
    from scratch_wadge_amd import problem as P
    from scratch_wadge_amd.adjoint import AdjointSolver, density_misfit, misfit_setup
    from scratch_wadge_amd.device import DeviceSolver
    prob = P.vortex2d_problem(n=32, N=3)
    dev = DeviceSolver(prob)
    Q0, _, target = misfit_setup(prob, dev, steps)
    adj = AdjointSolver(dev, checkpoint_every=ckpt)
    dev.run(4, fused=True, graph=True)              # warm-up, graph capture
    t_plain = _sync_time(lambda: dev.run(steps, fused=True, graph=True))
    adj.forward(Q0, 2 * ckpt)                       # warm-up, graph captures
    adj.backward(torch.zeros_like(Q0))
    out = {}
    t_fwd = _sync_time(lambda: out.setdefault("QT", adj.forward(Q0, steps)))
    QT = out["QT"].clone().requires_grad_(True)
    loss = density_misfit(prob, QT, target)
    loss.backward()
    loss = float(loss.detach())
    t_bwd = _sync_time(lambda: out.setdefault("g", adj.backward(QT.grad)))
    return {"workload": f"2D vortex 32x32x2 (K={prob.K}), N=3, {steps} steps, checkpoints every {ckpt}",
            "forward_ms": round(t_plain * 1e3, 2), "forward_with_checkpoints_ms": round(t_fwd * 1e3, 2),
            "adjoint_sweep_ms": round(t_bwd * 1e3, 2),
            "adjoint_over_forward": round(t_bwd / t_plain, 3),
            "forward_plus_adjoint_over_forward": round((t_fwd + t_bwd) / t_plain, 3),
            "loss": loss, "grad_norm": float(torch.linalg.norm(out["g"]))}


def n4_leg(n, steps=3):
    """The headline mesh at N = 4 (Np = 35, Nq = 44, Nf = 64): fused-stage launch
    time (HIP events, 5 steps after one warm-up step) and GDOF.stage/s."""
    import numpy as np
    import torch
    from scratch_wadge_amd import problem as P
    from scratch_wadge_amd import workmodel as W
    from scratch_wadge_amd.device import DeviceSolver
    prob = P.tgv3d_problem(n=n, N=4, curved=True)
    dev = DeviceSolver(prob)
    dev.step(prob.dt, fused=True)
    stream = torch.cuda.current_stream()
    evs = []
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        for s in range(5):
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record(stream)
            dev.stage_fused(s, prob.dt)
            b.record(stream)
            evs.append((a, b))
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms = float(np.mean([a.elapsed_time(b) for a, b in evs]))
    flops = W.stage_flops(3, prob.Nq, prob.Nf) * prob.K
    ok = bool(np.isfinite(dev.s["Q"].cpu().numpy()).all())
    del dev
    torch.cuda.empty_cache()
    return {"workload": f"3D TGV curved (warp 0.1) tets, {n}^3 x 6 = {prob.K} elements, N=4",
            "value": round(W.dofs(3, 4, prob.K) * 5 * steps / wall / 1e9, 4),
            "unit": "GDOF*stage/s", "stage_ms": round(ms, 4),
            "roofline": {"bound": "fp64 valu", "kernel": "stage_kernel",
                         "achieved": round(flops / (ms * 1e-3) / 1e12, 3),
                         "frac": round(flops / (ms * 1e-3) / 1e12 / W.FP64_PEAK_TFLOPS, 4),
                         "flops_per_element": W.stage_flops(3, prob.Nq, prob.Nf)},
            "finite": ok}


def main():
    args = parse()
    if args.copy_calibration > 0:
        copy_calibration(args.copy_calibration)
        return
    if args.gpus != 1:
        print(f"bench.py runs on one GPU: --gpus {args.gpus} is not supported (the element "
              f"partition across GPUs is designed but not built)", file=sys.stderr)
        sys.exit(2)
    if args.leg == "ensemble":
        print(json.dumps({"ensemble": ensemble_bench(args.ensemble_steps)}), flush=True)
        return
    if args.leg == "adjoint":
        print(json.dumps({"adjoint": adjoint_bench(args.adjoint_steps)}), flush=True)
        return
    if args.leg == "adjoint3d":
        print(json.dumps({"adjoint3d": adjoint3d_bench()}), flush=True)
        return
    import numpy as np
    import torch

    from scratch_wadge_amd import problem as P
    from scratch_wadge_amd import workmodel as W
    from scratch_wadge_amd.device import DeviceSolver

    t0 = time.perf_counter()
    prob = P.tgv3d_problem(n=args.n, N=args.N, curved=not args.affine)
    setup_s = time.perf_counter() - t0
    print(f"# setup K={prob.K} N={prob.N} Nq={prob.Nq} Nf={prob.Nf} in {setup_s:.1f}s",
          file=sys.stderr, flush=True)
    dev = DeviceSolver(prob)
    dt = prob.dt
    stream = torch.cuda.current_stream()

    def ev():
        e = torch.cuda.Event(enable_timing=True)
        e.record(stream)
        return e

    # ---- three-kernel path (the reference's rk_step structure): per-kernel times
    for _ in range(args.warmup):
        dev.step(dt)
    torch.cuda.synchronize()
    evs = []
    for _ in range(args.steps):
        for s in range(5):
            a = ev()
            dev.vol()
            b = ev()
            dev.surf()
            c = ev()
            dev.update(P.RK4A[s], P.RK4B[s], dt)
            evs.append((a, b, c, ev()))
    torch.cuda.synchronize()
    vol_ms = float(np.mean([a.elapsed_time(b) for a, b, c, d in evs]))
    surf_ms = float(np.mean([b.elapsed_time(c) for a, b, c, d in evs]))
    upd_ms = float(np.mean([c.elapsed_time(d) for a, b, c, d in evs]))
    split_stage_ms = float(np.mean([a.elapsed_time(d) for a, b, c, d in evs]))

    # ---- fused path (one launch per stage): the timed region for `value`
    dev.set_state(**prob.copy_state())
    for _ in range(args.warmup):
        dev.step(dt, fused=True)
    torch.cuda.synchronize()
    evf = []
    t_start = time.perf_counter()
    for _ in range(args.steps):
        for s in range(5):
            a = ev()
            dev.stage_fused(s, dt)
            evf.append((a, ev()))
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t_start
    stage_ms = float(np.mean([a.elapsed_time(b) for a, b in evf]))

    stages = 5 * args.steps
    value = W.dofs(prob.dim, prob.N, prob.K) * stages / elapsed / 1e9
    prof_file = (f"stage_kernel_tgv3d_{'affine' if args.affine else 'curved'}"
                 f"_K{prob.K}_N{prob.N}.md")
    prof = lambda key, kernel: profiled_value(key, kernel, prof_file)

    # 3D N = 3 runs a wave per face, the other shapes a team of lanes per element
    team = "team_" if (prob.dim, prob.N) == (3, 3) else ""
    stage_kernel, vol_kernel = team + "stage_kernel", team + "vol_kernel"

    def counter_tflops(kernel, ms):
        v = prof("fp64_lane_flops_per_launch", kernel)
        return None if v is None else round(v / (ms * 1e-3) / 1e12, 3)

    def prof_ms(kernel):
        v = prof("kernel_avg_us", kernel)
        return None if v is None else round(v / 1e3, 4)
    flops = W.stage_flops(prob.dim, prob.Nq, prob.Nf) * prob.K
    achieved = flops / (stage_ms * 1e-3) / 1e12
    vflops = W.vol_flops(prob.dim, prob.Nq, prob.Nf) * prob.K
    st = dev.get_state()
    varying_ms = None
    if args.extras:
        # ---- the same stage on a strongly varying state, where neighbouring nodes
        # differ beyond the log mean's series threshold (both branches taken); the
        # Taylor-Green state above takes the series branch throughout
        Qv, rqv, qfv = P.varying_state(prob, seed=7, amp=0.3)
        dev.set_state(Q=Qv, rhsQ=rqv, Qf=qfv, resQ=np.zeros_like(Qv))
        evr = []
        for _ in range(3):
            for s in range(5):
                a = ev()
                dev.stage_fused(s, dt)
                evr.append((a, ev()))
        torch.cuda.synchronize()
        varying_ms = float(np.mean([a.elapsed_time(b) for a, b in evr[5:]]))
        if not np.isfinite(dev.s["Q"].cpu().numpy()).all():
            print("# varying state is not finite after its steps", file=sys.stderr)
            sys.exit(1)
    if not all(np.isfinite(v).all() for v in st.values()):
        print("# state is not finite after the run", file=sys.stderr)
        sys.exit(1)

    out = {
        "metric": f"GDOF*RK-stage/s (3D {'affine' if args.affine else 'curved'} tet N={prob.N}, FP64)",
        "value": round(value, 4),
        "unit": "GDOF*stage/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(elapsed / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (Taylor-Green initial state on a generated warped periodic tet mesh)",
        "config": {"workload": f"3D TGV {'affine' if args.affine else 'curved (warp 0.1)'} tets, "
                               f"{args.n}^3 x 6 = {prob.K} elements, N={prob.N}",
                   "K": prob.K, "N": prob.N, "Np": prob.Np, "Nq": prob.Nq, "Nf": prob.Nf,
                   "stages_per_step": 5, "tau": prob.tau},
        "path": "fused stage kernel (vol+surf+update, one launch per RK stage)",
        "kernels_ms": {"stage_fused": round(stage_ms, 4), "split_stage": round(split_stage_ms, 4),
                       "vol": round(vol_ms, 4), "surf": round(surf_ms, 4), "update": round(upd_ms, 4)},
        "roofline": {
            "bound": "fp64 valu",
            "pipe": "FP64 vector ALU: the flux differencing (most of the flops) is "
                    "elementwise D o F over node pairs, not a matrix product; the "
                    "small dense operator products (lift, VqPq, face traces) run on "
                    "the FP64 matrix cores, whose dense peak equals the vector peak",
            "kernel": stage_kernel,
            "achieved": round(achieved, 3), "peak": W.FP64_PEAK_TFLOPS, "unit": "TFLOP/s",
            "frac": round(achieved / W.FP64_PEAK_TFLOPS, 4),
            "flops_per_launch": flops,
            "flops_per_element": W.stage_flops(prob.dim, prob.Nq, prob.Nf),
            "launch_ms": round(stage_ms, 4),
            "traffic": prof("traffic_bytes_per_launch", stage_kernel),
            "traffic_source": "rocprofv3 FETCH_SIZE x2.0 + WRITE_SIZE x1.0 (copy-calibrated), "
                              f"profiles/{prof_file}",
            "counter_tflops": counter_tflops(stage_kernel, stage_ms),
            "counter_source": "64 (ADD+MUL+TRANS) + 128 FMA FP64 instructions per launch "
                              f"(SQ_INSTS_VALU_*_F64), profiles/{prof_file}, over launch_ms; "
                              "vector ALU only, the matrix-core products are not in these counters",
            "profile_kernel_avg_ms": prof_ms(stage_kernel),
        },
        "vol_kernel_roofline": {"bound": "fp64 valu", "kernel": vol_kernel,
                                "achieved": round(vflops / (vol_ms * 1e-3) / 1e12, 3),
                                "frac": round(vflops / (vol_ms * 1e-3) / 1e12 / W.FP64_PEAK_TFLOPS, 4),
                                "flops_per_element": W.vol_flops(prob.dim, prob.Nq, prob.Nf),
                                "launch_ms": round(vol_ms, 4),
                                "counter_tflops": counter_tflops(vol_kernel, vol_ms),
                                "profile_kernel_avg_ms": prof_ms(vol_kernel)},
        "hbm_GBs": {
            "stage_fused": round(W.bytes_stage_fused(prob.dim, prob.Nq, prob.Nf) * prob.K / (stage_ms * 1e-3) / 1e9, 1),
            "surf": round(W.bytes_surf(prob.dim, prob.Nq, prob.Nf) * prob.K / (surf_ms * 1e-3) / 1e9, 1),
            "update": round(W.bytes_update(prob.dim, prob.Nq, prob.Nf) * prob.K / (upd_ms * 1e-3) / 1e9, 1),
        },
        "cpu_baseline": None,
    }
    if args.cpu:
        out["cpu_baseline"] = cpu_baseline(prob, args.cpu_seconds)
    if varying_ms is not None:
        out["varying_state"] = {
            "state": "density and pressure 1 + 0.3 sin(x.k + phase), velocities 0.5: both "
                     "log-mean branches (the Taylor-Green state takes the series branch at "
                     "every pair)",
            "stage_ms": round(varying_ms, 4),
            "value": round(W.dofs(prob.dim, prob.N, prob.K) / (varying_ms * 1e-3) / 1e9, 4),
            "frac": round(flops / (varying_ms * 1e-3) / 1e12 / W.FP64_PEAK_TFLOPS, 4)}
    if args.extras and args.N == 3 and not args.affine:
        del dev
        torch.cuda.empty_cache()
        out["N4"] = n4_leg(args.n)
        print(f"# N4 {out['N4']}", file=sys.stderr, flush=True)
    if args.extras:
        if "dev" in locals():
            del dev
        torch.cuda.empty_cache()
        out["ensemble"] = ensemble_bench(args.ensemble_steps)
        print(f"# ensemble {out['ensemble']}", file=sys.stderr, flush=True)
        out["adjoint"] = adjoint_bench(args.adjoint_steps)
        print(f"# adjoint {out['adjoint']}", file=sys.stderr, flush=True)
        torch.cuda.empty_cache()
        out["adjoint3d"] = adjoint3d_bench()
        print(f"# adjoint3d {out['adjoint3d']}", file=sys.stderr, flush=True)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
