"""The initial projection u(VqPq v(Q)), u(VfPq v(Q)) in one launch against the same
maps as FP64 tensor operations on the CPU: every shape, one element, full and partly
filled last workgroups, on a rough state.  Nothing beyond K elements is written."""

import numpy as np
import pytest
import torch

import torch_ref as TR
from helpers import has_rule, relerr, small_problem
from scratch_wadge_amd import problem as P

pytestmark = pytest.mark.gpu

SHAPES = [(d, N) for d in (2, 3) for N in range(1, 6) if has_rule(d, N)]


@pytest.mark.parametrize("dim,N", SHAPES)
def test_projection(dim, N):
    from scratch_wadge_amd.device import DeviceSolver, _ptr
    prob = small_problem(dim, N)
    Q, _, _ = P.varying_state(prob, seed=6, amp=0.05)
    ref = [t.numpy().reshape(prob.K, -1) for t in TR.project(TR.Ops(prob, "cpu"), torch.as_tensor(Q))]
    sv = DeviceSolver(prob)
    Qd = torch.as_tensor(Q, device="cuda").reshape(-1).contiguous()
    for K in sorted({1, 2, prob.K // 2 + 1, prob.K - 1, prob.K}):
        print(f"case project dim={dim} N={N} K={K}", flush=True)
        uq, uf = torch.full_like(sv.s["rhsQ"], -7.0), torch.full_like(sv.s["Qf"], -7.0)
        sv.plan.project(K, _ptr(sv.c["VqPq"]), _ptr(sv.c["VfPq"]), _ptr(Qd), _ptr(uq), _ptr(uf), sv.stream())
        for t, r in zip((uq, uf), ref):
            t = t.cpu().numpy().reshape(prob.K, -1)
            # both sides: a sum of at most 44 products between maps of condition ~ 1e2
            assert relerr(t[:K], r[:K]) < 1e-13
            assert np.all(t[K:] == -7.0)


def test_refused_states():
    from scratch_wadge_amd.adjoint import AdjointSolver
    from scratch_wadge_amd.device import DeviceSolver
    prob = small_problem(2, 2)
    adj = AdjointSolver(DeviceSolver(prob))
    Q = torch.as_tensor(prob.Q, device="cuda").reshape(-1)
    with pytest.raises(RuntimeError):
        adj.forward(Q.float(), 1)
    with pytest.raises(RuntimeError):
        adj.forward(Q[:-1], 1)
