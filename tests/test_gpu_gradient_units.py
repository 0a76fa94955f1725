"""Gradients in other units: lengths times 2^k and primitives times 2^j scale every
operation of the gradients and their limiter exactly, so the gradients times
2^(k - j) are the same bits, inside, at and past the ranges of the fast quotients
(cells of 2^-66 to 2^50 in 3D, primitives of 2^-240 to 2^150)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("k,j", [(-50, 0), (-60, -180), (-64, 100), (40, -200), (48, 140),
                                 (54, 0), (-72, 0), (0, -260), (10, 170)])
@pytest.mark.parametrize("name,n", [("kh_2d", 30), ("kh_2d", 190), ("sedov_3d", 11), ("sedov_3d", 30)])
def test_gradients_scale_with_the_units(gpu, name, n, k, j, limiter):
    from phd import problems
    print("case units %s n=%d 2^%d 2^%d limiter %d" % (name, n, k, j, limiter), flush=True)
    p = problems.PROBLEMS[name](n=n, seed=1)
    pc, mesh, dim = p.particles, p.mesh, p.dim
    rng = np.random.default_rng(n)
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, pc.get_carray_size())
        pc[f][:] = torch.as_tensor(v if q in (0, dim + 1) else v - 1.2, device=gpu)
    p.recon.slope_limiter = limiter
    real = pc["tag"] == 0
    p.recon.compute_gradients(pc, mesh, p.domain_manager)
    want = p.recon.grad.rows()[real].clone()
    g, fg = pc.carray_named_groups, mesh.faces.carray_named_groups
    for f in g["position"] + g["dcom"]:
        pc[f][:] *= 2.0 ** k
    for f in fg["com"]:
        mesh.faces[f][:] *= 2.0 ** k
    mesh.faces["area"][:] *= 2.0 ** (k * (dim - 1))
    pc["volume"][:] *= 2.0 ** (k * dim)
    for f in g["primitive"]:
        pc[f][:] *= 2.0 ** j
    mesh.invalidate_plan()
    p.recon.compute_gradients(pc, mesh, p.domain_manager)
    got = p.recon.grad.rows()[real] * 2.0 ** (k - j)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    assert torch.equal(got, want), int((got != want).sum())
