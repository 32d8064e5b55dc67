"""The lazily taken logarithms of the volume term and of its VJP: waves whose volume
nodes are smooth but whose face traces are not, and the reverse, must take the
log-mean branches of the oracle and of the reference gradient."""

import numpy as np
import pytest

from helpers import relerr, small_problem

pytestmark = pytest.mark.gpu

# Every sum of at most 2 (Nq + Nf) terms of a few rounded operations each: the
# parity bar of the volume and surface terms.
TOL = 1e-12


ROUGH = ["volume", "faces", "one face point", "one volume node"]


def rough_rhs_state(prob, rough, rng):
    """Projected volume states and traces, near-uniform but for the rough ones."""
    dim, nf = prob.dim, prob.nfields

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
    return uq.reshape(-1), uf.reshape(-1)


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4)])
@pytest.mark.parametrize("rough", ROUGH)
def test_rhs_with_rough_volume_or_traces(oracle, dim, N, rough):
    from scratch_wadge_amd.device import DeviceSolver
    prob = small_problem(dim, N)
    rng = np.random.default_rng(dim * 10 + N)
    uq, uf = rough_rhs_state(prob, rough, rng)
    print(f"case lazy logs dim={dim} N={N} rough={rough} K={prob.K}", flush=True)
    r_gpu, _ = DeviceSolver(prob).rhs(uq, uf)
    r_ref, _ = oracle.rhs(prob, uq, uf)
    e = relerr(r_gpu, r_ref)
    print(f"rel L2 {e:.2e}", flush=True)
    assert e < TOL


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 3), (2, 4), (3, 2), (3, 3), (3, 4)])
@pytest.mark.parametrize("rough", ROUGH)
def test_rhs_vjp_with_rough_volume_or_traces(dim, N, rough):
    import torch
    import torch_ref as TR
    from scratch_wadge_amd.device import DeviceSolver, _ptr
    prob = small_problem(dim, N)
    rng = np.random.default_rng(dim * 10 + N)
    uq, uf = rough_rhs_state(prob, rough, rng)
    print(f"case lazy logs vjp dim={dim} N={N} rough={rough} K={prob.K}", flush=True)
    dev = DeviceSolver(prob)
    D = lambda x: torch.as_tensor(x, dtype=torch.float64, device="cuda:0")
    c, uqd, ufd, Rb = dev.c, D(uq), D(uf), D(rng.standard_normal(uq.shape))
    sbar, uqb, ufb = torch.empty_like(ufd), torch.empty_like(uqd), torch.empty_like(ufd)
    dev.plan.rhs_vjp(prob.K, *(_ptr(c[x]) for x in ("vgeo", "vfgeo", "fgeo", "mapPq", "nrJ", "nsJ", "ntJ",
                                                    "Drq", "Dsq", "Dtq", "VqLq", "VfPq")),
                     _ptr(uqd), _ptr(ufd), _ptr(Rb), _ptr(sbar), _ptr(uqb), _ptr(ufb), dev.stream())
    a, b = uqd.clone().requires_grad_(True), ufd.clone().requires_grad_(True)
    (TR.rhs(TR.Ops(prob, "cuda:0"), a, b) * Rb).sum().backward()
    torch.cuda.synchronize()
    e = [relerr(x.cpu().numpy(), y.cpu().numpy()) for x, y in ((uqb, a.grad), (ufb, b.grad))]
    print("rel L2", e, flush=True)
    # the bar of the VJP against the reference gradient: ten times the forward bar (a
    # derivative of the log branch divides by the difference of the logarithms)
    assert max(e) < 10 * TOL
