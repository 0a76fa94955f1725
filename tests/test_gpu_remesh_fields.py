"""GPU check of Mesh.build_geometry on particle containers with fields of every
type, with and without the groups of the step: ghosts take every field from
their images."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [True, False])
def test_ghosts_take_every_field(gpu, groups):
    from phd import problems
    prob = problems.PROBLEMS["sod_2d"](n=9, seed=2)
    pc, mesh = prob.particles, prob.mesh
    n = pc.get_carray_size()
    for k, dtype in enumerate(("int", "long", "longlong", "double")):
        pc.register_carray(n, "extra-" + dtype, dtype)
        pc["extra-" + dtype][:] = torch.arange(n, device=gpu) % (100 + k)
    if not groups:
        del pc.carray_named_groups["primitive"], pc.carray_named_groups["conservative"]
    mesh.build_geometry(pc, prob.domain_manager)
    tag, image = pc["tag"].cpu().numpy(), pc["map"].cpu().numpy()
    ghosts = np.nonzero(tag)[0]
    assert ghosts.size
    for f in ["density", "pressure", "mass", "energy"] + \
            ["extra-" + d for d in ("int", "long", "longlong", "double")]:
        v = pc[f].cpu().numpy()
        assert np.array_equal(v[ghosts], v[image[ghosts]]), f
    assert (pc["type"].cpu().numpy()[ghosts] == 2).all()
