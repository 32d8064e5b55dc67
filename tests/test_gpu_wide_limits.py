"""Where the fused stage changes its launch: the largest meshes of the two launches for
small meshes and the ones just above, on a curved or perturbed mesh of each shape, equal
bit for bit to the packed stage that ensembles run.  The plan's limits say which launch a
mesh takes, so that the comparison cannot quietly be one of the packed stage with itself."""

import numpy as np
import pytest
import torch

from helpers import has_rule
from scratch_wadge_amd import _lib
from scratch_wadge_amd import problem as P

pytestmark = pytest.mark.gpu

SHAPES = [(d, N) for d in (2, 3) for N in range(1, 6) if has_rule(d, N)]
ONE_LAUNCH = (3, 3)          # a wave per face for every mesh


def limits(dim, N):
    o = P.vortex2d_problem(n=3, N=N) if dim == 2 else P.tgv3d_problem(n=3, N=N, curved=False)
    plan = _lib.Plan(dim, N, o.Nq, o.Nfq, o.gamma, o.tau)
    return plan.wide_limits()


@pytest.mark.parametrize("dim,N", SHAPES)
def test_limits(dim, N):
    small, large = limits(dim, N)
    if (dim, N) == ONE_LAUNCH:
        assert (small, large) == (0, 0)
        return
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    # up to two elements per CU; at least as many where every workgroup is resident
    assert 0 < small <= 2 * cus and small <= large and large % cus == 0


# meshes of tests that take the wide launches for granted: cells per side and which launch
@pytest.mark.parametrize("dim,N,n,large", [
    (2, 1, 4, False), (2, 1, 33, True), (2, 2, 4, False), (2, 2, 33, True), (2, 3, 4, False),
    (2, 3, 29, True), (2, 4, 4, False), (2, 4, 29, True), (2, 5, 4, False), (2, 5, 19, True),
    (3, 1, 3, False), (3, 1, 6, True), (3, 2, 3, False), (3, 2, 5, True), (3, 4, 3, False),
    (3, 4, 5, True)])
def test_meshes_of_both_launches(dim, N, n, large):
    K = 2 * n * n if dim == 2 else 6 * n ** 3
    lo, hi = limits(dim, N)
    assert (lo < K <= hi) if large else K <= lo


@pytest.mark.parametrize("dim,N", [s for s in SHAPES if s != ONE_LAUNCH])
def test_stage_at_the_limits(dim, N):
    from scratch_wadge_amd.device import DeviceSolver, _ptr
    from scratch_wadge_amd.ensemble import group_of
    small, large = limits(dim, N)
    n = int(np.ceil(np.sqrt((large + 1) / 2))) if dim == 2 else int(np.ceil(np.cbrt((large + 1) / 6)))
    prob = P.vortex2d_problem(n=n, N=N, beta=1.0) if dim == 2 else P.tgv3d_problem(n=n, N=N, curved=True)
    assert prob.K > large
    Q, uq, uf = P.varying_state(prob, seed=4, amp=0.1 if dim == 2 else 0.03)
    for K in (small, small + 1, large, large + 1):
        print(f"case wide limits dim={dim} N={N} K={K} of {prob.K}", flush=True)
        a, b = DeviceSolver(prob), DeviceSolver(prob)
        for sv in (a, b):
            sv.set_state(Q=Q, rhsQ=uq, Qf=uf)
            sv.Qf_alt.copy_(sv.s["Qf"])
        g = group_of(b)
        g.K, g.dt = K, 0.1 * prob.dt
        batch = _lib.Batch(dim, [g], prob.gamma, prob.tau, b.stream())
        c, s = a.c, a.s
        geo = [_ptr(c[x]) for x in ("vgeo", "vfgeo", "fgeo", "mapPq", "nrJ", "nsJ", "ntJ", "Drq", "Dsq",
                                    "Dtq", "VqLq", "VqPq", "VfPq", "Jq")]
        a.plan.stage(K, *geo, P.RK4A[1], P.RK4B[1], g.dt, _ptr(s["Qf"]), _ptr(a.Qf_alt), _ptr(s["rhsQ"]),
                     _ptr(s["resQ"]), _ptr(s["Q"]), a.stream())
        batch.stage(P.RK4A[1], P.RK4B[1], b.stream())
        torch.cuda.synchronize()
        for x in ("Q", "resQ", "rhsQ"):
            assert torch.equal(s[x], b.s[x]), (K, x)
        assert torch.equal(a.Qf_alt, b.Qf_alt), K
        batch.close()
