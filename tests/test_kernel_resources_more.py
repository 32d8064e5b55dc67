"""Register budget of the kernels that test_kernel_resources.py does not name, from the
same resource remarks: the fused stage of small meshes, the projections and the VJP
kernels of every shape must not spill to scratch, and the wave-per-face kernels of 3D
N = 3 must keep the three waves per SIMD that their shared LDS tile is made for.  A wave
of the RHS VJP alone on its SIMD has nothing to hide its latencies behind: two."""

from test_kernel_resources import _shape, remarks  # noqa: F401  (a fixture)

KERNELS = {"stage_wide": 12, "project_kernel": 9, "proj_vjp_kernel": 9, "rhs_vjp_kernel": 9,
           "update_vjp_kernel": 4, "update_vjp_mfma_kernel": 5}


def test_small_mesh_and_adjoint_kernels_do_not_spill(remarks):  # noqa: F811
    for kernel, count in KERNELS.items():
        found = {n: r for n, r in remarks.items() if f"{len(kernel)}{kernel}" in n}
        assert len(found) == count, (kernel, len(found))
        for name, r in found.items():
            assert r.get("ScratchSize", 0) == 0, (name[:90], r)


def test_wave_per_face_kernels_keep_three_waves(remarks):  # noqa: F811
    for kernel in ("team_stage_kernel", "team_vol_kernel"):
        (r,) = [r for n, r in remarks.items() if kernel in n and _shape(n) == (3, 23, 12)]
        assert r["Occupancy"] >= 3, (kernel, r)


def test_rhs_vjp_keeps_two_waves(remarks):  # noqa: F811
    found = {_shape(n): r for n, r in remarks.items() if "rhs_vjp_kernel" in n}
    assert len(found) == 9
    for shape, r in found.items():
        assert r["Occupancy"] >= 2, (shape, r)
