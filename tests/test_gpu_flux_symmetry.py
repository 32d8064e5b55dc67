"""The two elements of a face take the same numerical flux, bit for bit: the surface
kernel's values at matching face points cancel exactly, also where the log means take
their logarithm branch (rough states).  Two elements are matched point by point with
opposite normals, and an operator of unit rows stands in for the lift, so that rows of
the result are single face values."""

import numpy as np
import pytest
import torch

from helpers import small_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
@pytest.mark.parametrize("amp", [1e-3, 0.05, 0.8])
def test_face_values_cancel(dim, N, amp):
    from scratch_wadge_amd import _lib
    prob = small_problem(dim, N)
    Nq, Nf, nf = prob.Nq, prob.Nf, dim + 2
    rng = np.random.default_rng(100 * dim + N)
    pairs = 64
    K = 2 * pairs
    rho = np.exp(amp * rng.uniform(-1, 1, (K, Nf)))
    p = np.exp(amp * rng.uniform(-1, 1, (K, Nf)))
    vel = rng.standard_normal((K, dim, Nf))
    U = np.empty((K, nf, Nf))
    U[:, 0] = rho
    U[:, 1:-1] = rho[:, None] * vel
    U[:, -1] = p / (prob.gamma - 1.0) + 0.5 * rho * (vel ** 2).sum(1)
    # element 2 q and 2 q + 1 meet at every face point, normals opposite
    mate = np.arange(K) ^ 1
    mapP = (mate[:, None] * Nf * nf + np.arange(Nf)[None, :]).astype(np.int32)
    g = np.empty((K, dim + 1, Nf))
    g[:, :dim] = rng.standard_normal((K, dim, Nf))
    g[:, dim] = np.sqrt((g[:, :dim] ** 2).sum(1))
    g[1::2, :dim], g[1::2, dim] = -g[0::2, :dim], g[0::2, dim]

    D = lambda a: torch.as_tensor(np.ascontiguousarray(a).reshape(-1), device="cuda")
    plan = _lib.Plan(dim, N, Nq, prob.Nfq, prob.gamma, 1.0)
    Qf, fgeo, mapPq, zero = D(U), D(g), D(mapP), torch.zeros(K * nf * Nf, dtype=torch.float64, device="cuda")
    print(f"case flux symmetry dim={dim} N={N} amp={amp}", flush=True)
    for c in range(0, Nf, Nq):
        n = min(Nq, Nf - c)
        L = np.zeros((Nf, Nq))                       # VqLq[i + f Nq]: row i takes face point c + i
        L[c + np.arange(n), np.arange(n)] = 1.0
        Ld, out = D(L), torch.zeros(K * nf * Nq, dtype=torch.float64, device="cuda")
        plan.surf(K, *(t.data_ptr() for t in (fgeo, mapPq, Ld, Qf, zero, out)),
                  torch.cuda.current_stream().cuda_stream)
        v = out.cpu().numpy().reshape(K, nf, Nq)[:, :, :n]
        assert np.isfinite(v).all() and np.abs(v).min(axis=(0, 2)).max() > 0
        assert np.array_equal(v[0::2], -v[1::2])
