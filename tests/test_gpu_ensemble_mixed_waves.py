"""Ensemble launches whose workgroups hold waves of every kind side by side: smooth
ones (no logarithms), ones with rough volume states, ones with rough traces only, and
idle padding past a problem's last element.  A wave's arithmetic must not depend on its
neighbours: the widths of two and four waves give the bits of the one-wave launch."""

import numpy as np
import pytest

from helpers import has_rule, small_problem
from scratch_wadge_amd import problem as P

pytestmark = pytest.mark.gpu


def mixed_state(prob, seed):
    """Near-uniform projected states and traces; by tiles of a wave's elements in turn
    rough in the volume, rough on the faces, smooth."""
    rng = np.random.default_rng(seed)
    per_wave = 64 // (12 if prob.Nq == 23 else prob.Nq)
    kind = np.arange(prob.K) // per_wave % 3

    def state(npts, rough):
        U = np.empty((prob.K, prob.nfields, npts))
        U[:, 0] = 1.0 + 1e-4 * rng.standard_normal((prob.K, npts))
        vel = 0.3 + 1e-3 * rng.standard_normal((prob.K, prob.dim, npts))
        U[:, 1:-1] = U[:, :1] * vel
        U[:, -1] = 2.5 + 0.5 * U[:, 0] * (vel ** 2).sum(1)
        U[rough] *= rng.uniform(0.8, 1.25, size=(int(rough.sum()), 1, npts))
        return U.reshape(-1)

    return dict(Q=state(prob.Nq, kind == 0), rhsQ=state(prob.Nq, kind == 0),
                Qf=state(prob.Nf, kind == 1))


def problems(dim):
    """Every degree; element counts that fill no workgroup of two or four waves."""
    out = []
    for N in range(1, 6):
        if has_rule(dim, N):
            p = (P.vortex2d_problem(n=9, N=N, perturb=0.05, seed=N) if dim == 2
                 else small_problem(3, N))
            out.append((p, mixed_state(p, 10 * dim + N)))
    return out


@pytest.mark.parametrize("dim,widths", [(2, (2, 4)), (3, (2,))])
def test_widths_give_the_bits_of_one_wave(dim, widths):
    from scratch_wadge_amd.ensemble import Ensemble
    probs = problems(dim)
    runs = {}
    for W in (1,) + widths:
        print(f"case mixed waves dim={dim} W={W}", flush=True)
        ens = Ensemble([p for p, _ in probs])
        for sv, (_, s) in zip(ens.solvers, probs):
            sv.set_state(**s)
        ens.set_config(grid=0, waves_per_group=W)
        assert ens.config()["waves_per_group"] == W
        for stage in range(2):
            ens.batch.stage(P.RK4A[stage], 0.01 * P.RK4B[stage], ens.stream())
        runs[W] = [ens.state(q) for q in range(len(probs))]
        ens.close()
    for q, (p, _) in enumerate(probs):
        for f, one in runs[1][q].items():
            assert np.isfinite(one).all(), (dim, p.N, f)
            for W in widths:
                assert np.array_equal(runs[W][q][f], one), (dim, p.N, f, W)
