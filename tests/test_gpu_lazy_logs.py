"""The lazily taken logarithms of the volume term: waves whose volume nodes are
smooth but whose face traces are not, and the reverse, must take the log-mean
branches of the oracle."""

import numpy as np
import pytest

from helpers import relerr, small_problem

pytestmark = pytest.mark.gpu

# Every sum of at most 2 (Nq + Nf) terms of a few rounded operations each: the
# parity bar of the volume and surface terms.
TOL = 1e-12


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
@pytest.mark.parametrize("rough", ["volume", "faces", "one face point", "one volume node"])
def test_rhs_with_rough_volume_or_traces(oracle, dim, N, rough):
    from scratch_wadge_amd.device import DeviceSolver
    prob = small_problem(dim, N)
    rng = np.random.default_rng(dim * 10 + N)
    nf = prob.nfields

    def state(npts):
        """Near-uniform conservative state (density and pressure within 1e-4)."""
        U = np.empty((prob.K, nf, npts))
        U[:, 0] = 1.0 + 1e-4 * rng.standard_normal((prob.K, npts))
        vel = 0.3 + 1e-3 * rng.standard_normal((prob.K, dim, npts))
        U[:, 1:-1] = U[:, :1] * vel
        U[:, -1] = 2.5 + 1e-4 * rng.standard_normal((prob.K, npts)) + 0.5 * U[:, 0] * (vel ** 2).sum(1)
        return U

    def roughen(U):
        """Density and total energy of the same points scaled by 0.7 .. 1.3."""
        f = rng.uniform(0.7, 1.3, size=U[:, :1].shape)
        U *= f
        return U

    uq, uf = state(prob.Nq), state(prob.Nf)
    if rough == "volume":
        roughen(uq)
    elif rough == "faces":
        roughen(uf)
    elif rough == "one face point":
        uf[1::3, :, -1] *= 1.2
    else:
        uq[2::5, :, prob.Nq // 2] *= 1.2
    uq, uf = uq.reshape(-1), uf.reshape(-1)
    print(f"case lazy logs dim={dim} N={N} rough={rough} K={prob.K}", flush=True)
    r_gpu, _ = DeviceSolver(prob).rhs(uq, uf)
    r_ref, _ = oracle.rhs(prob, uq, uf)
    e = relerr(r_gpu, r_ref)
    print(f"rel L2 {e:.2e}", flush=True)
    assert e < TOL
