"""The fused stage of small meshes (an element's pairs spread over a workgroup), and
of 3D N = 3 on every mesh (a wave per face), against the packed one, which
ensembles run whatever their size: equal bit for bit for every shape, on meshes of
both launch shapes, with full and partly filled last workgroups, on the initial
state and on a state with both log-mean branches."""

import numpy as np
import pytest
import torch

from scratch_wadge_amd import _lib
from scratch_wadge_amd import problem as P

pytestmark = pytest.mark.gpu

# (dim, N, cells per side): 2 n^2 triangles, 6 n^3 tetrahedra.  The second mesh of
# each shape has more than two elements per CU of a 256-CU device and is still
# resident at once (750 of the 768 elements at 3D N = 4).
MESHES = [(2, 1, 4), (2, 1, 33), (2, 2, 4), (2, 2, 33), (2, 3, 4), (2, 3, 29), (2, 4, 4), (2, 4, 29),
          (2, 5, 4), (2, 5, 19), (3, 1, 3), (3, 1, 6), (3, 2, 3), (3, 2, 5), (3, 3, 3), (3, 3, 5),
          (3, 4, 3), (3, 4, 5)]


@pytest.mark.parametrize("dim,N,n", MESHES)
@pytest.mark.parametrize("state", ["ic", "varying"])
def test_stage_equals_packed_stage(dim, N, n, state):
    from scratch_wadge_amd.device import DeviceSolver, _ptr
    from scratch_wadge_amd.ensemble import group_of
    prob = P.vortex2d_problem(n=n, N=N, beta=1.0) if dim == 2 else P.tgv3d_problem(n=n, N=N, curved=True)
    dt = 0.1 * prob.dt
    arrays = {}
    if state == "varying":
        Q, uq, uf = P.varying_state(prob, seed=4, amp=0.1 if dim == 2 and n > 4 else 0.03)
        arrays = dict(Q=Q, rhsQ=uq, Qf=uf)
    for K in (prob.K, prob.K - 1, 1):
        print(f"case wide stage dim={dim} N={N} K={K} of {prob.K} {state}", flush=True)
        a, b = DeviceSolver(prob), DeviceSolver(prob)
        for sv in (a, b):
            sv.set_state(**arrays)
            sv.Qf_alt.copy_(sv.s["Qf"])       # traces beyond K stay as they are
        c, s = a.c, a.s
        geo = [_ptr(c[x]) for x in ("vgeo", "vfgeo", "fgeo", "mapPq", "nrJ", "nsJ", "ntJ", "Drq", "Dsq",
                                    "Dtq", "VqLq", "VqPq", "VfPq", "Jq")]
        g = group_of(b)
        g.K, g.dt = K, dt
        batch = _lib.Batch(dim, [g], prob.gamma, prob.tau)
        bufs = (b.s["Qf"], b.Qf_alt)
        for k in range(2):
            a.plan.stage(K, *geo, P.RK4A[k], P.RK4B[k], dt, _ptr(s["Qf"]), _ptr(a.Qf_alt), _ptr(s["rhsQ"]),
                         _ptr(s["resQ"]), _ptr(s["Q"]), a.stream())
            s["Qf"], a.Qf_alt = a.Qf_alt, s["Qf"]
            batch.stage(P.RK4A[k], P.RK4B[k])
        torch.cuda.synchronize()
        for x in ("Q", "resQ", "rhsQ"):
            assert torch.equal(s[x], b.s[x]), x
        assert torch.equal(s["Qf"], bufs[batch.current()])
        assert np.isfinite(s["Q"].cpu().numpy()).all()
        batch.close()
