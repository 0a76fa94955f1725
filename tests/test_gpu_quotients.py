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


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("scale", [0, 60, 99, 130, 300])
@pytest.mark.parametrize("name,n", [("kh_2d", 33), ("sod_2d", 4), ("sedov_3d", 11)])
def test_gradients_equal_oracle_over_scales(gpu, name, n, scale, limiter):
    """Primitives in and past the ranges Shared takes, zeros among them, in a
    third of the windows' cells: the limited gradients bit for bit."""
    from oracle import oracle
    from phd import problems
    from parity import assert_bitwise
    print("case gradients %s n=%d scale 2^+-%d limiter %d" % (name, n, scale, limiter), flush=True)
    p = problems.PROBLEMS[name](n=n, seed=1)
    pc = p.particles
    na = pc.get_carray_size()
    rng = np.random.default_rng(scale + n)
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, na) if q in (0, p.dim + 1) else rng.normal(0, 1, na)
        some = rng.random(na) < 0.01
        v[some] *= 2.0 ** rng.integers(-scale, scale + 1, some.sum())
        v[rng.random(na) < 0.05] = 0.0
        pc[f][:] = torch.as_tensor(v, device=gpu)
    a = problems.host_arrays(p)
    p.recon.slope_limiter = limiter
    p.recon.compute_gradients(pc, p.mesh, p.domain_manager)
    grad, rc, _ = oracle.compute_gradients(a, limiter)
    assert rc == 0
    real = a["tag"] == 0
    got = p.recon.grad.rows().cpu().numpy()
    for q in range(len(grad)):
        assert_bitwise(got[real, q], grad[q][real], "grad %d" % q)
