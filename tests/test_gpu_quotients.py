"""The fused face kernel's Shared arithmetic (2D) against the operators on the
GPU: the same fluxes from phd_face_flux and from the materialised states and
the stand-alone solver, which use / and sqrt, bit for bit, over magnitudes
inside, at and past the ranges Shared takes."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0, 40, 99, 104])
@pytest.mark.parametrize("dim,n", [(2, 37), (3, 9)])
def test_fused_fluxes_equal_materialised(gpu, dim, n, scale):
    import phd
    from phd import _native as nat, problems
    from phd.views import cells_view, faces_view
    print("case dim %d n %d scale 2^+-%d" % (dim, n, scale), flush=True)
    p = (problems.kh_2d if dim == 2 else problems.sedov_3d)(n=n)
    pc, mesh = p.particles, p.mesh
    rng = np.random.default_rng(scale + dim)
    na = pc.get_carray_size()
    nf = mesh.faces.get_carray_size()

    def put(t, v):
        t[:] = torch.as_tensor(v, device=t.device)
    g = pc.carray_named_groups
    two = 2.0 ** rng.integers(-scale, scale + 1, (dim + 2, na))
    for q, f in enumerate(g["primitive"]):
        v = np.exp(rng.uniform(-1, 1, na)) if q in (0, dim + 1) else rng.normal(0, 1, na)
        v *= two[q]
        if 0 < q < dim + 1:
            v[rng.random(na) < 0.2] = 0.0
        put(pc[f], v)
    for f in mesh.faces.carray_named_groups["velocity"]:
        put(mesh.faces[f], rng.normal(0, 0.2, nf))
    lib, h = nat.flux(), nat.handle()
    recon = p.recon
    recon.compute_gradients(pc, mesh, p.domain_manager, check_errors=False)
    rec = recon.grad.data
    rec[:, dim + 2:dim + 2 + dim * (dim + 2)] *= torch.as_tensor(
        2.0 ** rng.integers(-scale, scale + 1, (na, 1)), device=rec.device)
    names = g["primitive"]
    c, fv = cells_view(pc), faces_view(mesh)

    def arrays():
        return [torch.zeros(nf, dtype=torch.float64, device=rec.device) for _ in names]
    for solver in (nat.SOLVER_HLLC, nat.SOLVER_HLL):
        for boost in (0, 1):
            for gizmo in (0, 1):
                L, R, A, B = arrays(), arrays(), arrays(), arrays()
                args = (rec.data_ptr(), recon.grad.ld, 1.4, 1e-3, boost, gizmo, nat.ORDER_LINEAR)
                nat.check(lib.phd_compute_states(
                    h, mesh.plan(pc), ctypes.byref(c), ctypes.byref(fv), *args,
                    nat.STAGE_SPATIAL | nat.STAGE_TEMPORAL, nat.ptr_array(L), nat.ptr_array(R)),
                    "phd_compute_states")
                nat.check(lib.phd_compute_fluxes(h, ctypes.byref(fv), dim, nat.ptr_array(L),
                                                 nat.ptr_array(R), 1.4, boost, solver,
                                                 nat.ptr_array(A)), "phd_compute_fluxes")
                nat.check(lib.phd_face_flux(h, mesh.plan(pc), ctypes.byref(c), ctypes.byref(fv),
                                            *args, solver, nat.ptr_array(B)), "phd_face_flux")
                for q, (x, y) in enumerate(zip(A, B)):
                    x, y = x.cpu().numpy(), y.cpu().numpy()
                    same = (x.view(np.int64) == y.view(np.int64)) | (np.isnan(x) & np.isnan(y))
                    assert same.all(), (solver, boost, gizmo, q, int((~same).sum()))
