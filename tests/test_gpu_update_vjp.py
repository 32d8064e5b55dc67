"""The update VJP (products on MFMA or a lane per row, by shape) against autograd of the
reference update on the CPU: every shape, one element, full and partly filled last
workgroups.  Nothing beyond K elements is written."""

import numpy as np
import pytest
import torch

import torch_ref as TR
from helpers import has_rule, relerr, small_problem
from scratch_wadge_amd import problem as P

pytestmark = pytest.mark.gpu

SHAPES = [(d, N) for d in (2, 3) for N in range(1, 6) if has_rule(d, N)]


@pytest.mark.parametrize("dim,N", SHAPES)
def test_update_vjp_matches_reference_gradient(dim, N):
    from scratch_wadge_amd.device import DeviceSolver, _ptr
    prob = small_problem(dim, N)
    rng = np.random.default_rng(8)
    Q, _, _ = P.varying_state(prob, seed=6, amp=0.05)
    fa, fb, dt = P.RK4A[3], P.RK4B[3], 2e-3
    rand = lambda n: torch.as_tensor(rng.standard_normal(n))
    nq, nf = prob.Q.size, prob.Qf.size
    bars = [rand(nq), rand(nq), rand(nq), rand(nf)]             # of Q', res', rhsQ', Qf'
    ins = [t.requires_grad_() for t in (0.1 * rand(nq), 1e-3 * rand(nq), torch.as_tensor(Q).clone())]
    outs = TR.update(TR.Ops(prob, "cpu"), fa, fb, dt, *ins)
    ref = torch.autograd.grad(outs, ins, bars)                   # R, res, Q
    sv = DeviceSolver(prob)
    Qo = outs[0].detach().cuda()
    for K in sorted({1, 2, prob.K // 2 + 1, prob.K - 1, prob.K}):
        print(f"case update vjp dim={dim} N={N} K={K}", flush=True)
        Qb, rb, uqb, ufb = [t.cuda() for t in bars]
        Rb = torch.full_like(Qb, -7.0)
        sv.plan.update_vjp(K, _ptr(sv.c["Jq"]), _ptr(sv.c["VqPq"]), _ptr(sv.c["VfPq"]), fa, fb, dt,
                           _ptr(Qo), _ptr(Qb), _ptr(rb), _ptr(uqb), _ptr(ufb), _ptr(Rb), sv.stream())
        for t, r, kept in zip((Rb, rb, Qb), ref, (torch.full_like(bars[0], -7.0), bars[1], bars[0])):
            t, r, kept = (x.cpu().numpy().reshape(prob.K, -1) for x in (t, r, kept))
            # eight products of at most 64 terms around maps of condition ~ 1e3; the
            # projection is idempotent to 1e-14
            assert relerr(t[:K], r[:K]) < 1e-11
            assert np.array_equal(t[K:], kept[K:])
