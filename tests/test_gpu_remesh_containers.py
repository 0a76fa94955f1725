"""GPU check of Mesh.build_geometry on containers that the step's kernels do not
take whole: more primitive or conservative fields than a cells view holds,
groups naming fields that are not there, arrays that are views with a stride, a
wide map, and a domain manager with only the members the mesh reads.  The ghosts
take every field from their images and the mesh is that of the plain container."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(dim):
    from phd import problems
    return problems.PROBLEMS["sod_2d" if dim == 2 else "sedov_3d"](n=9 if dim == 2 else 5, seed=2)


class Box(object):
    """What build_geometry reads of a domain manager."""

    def __init__(self, dm):
        self.xmin, self.xmax, self.boundary_condition = dm.xmin, dm.xmax, dm.boundary_condition


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("how", ["plain", "scalars", "missing", "strided", "wide_map", "box"])
def test_ghosts_of_unusual_containers(gpu, dim, how):
    print("case re-mesh %s dim %d" % (how, dim), flush=True)
    prob, plain = _problem(dim), _problem(dim)
    pc, domain = prob.particles, prob.domain_manager
    fields = ["density", "pressure", "mass", "energy", "ids"]
    if how == "scalars":
        for f, group in (("dye", "primitive"), ("dye2", "primitive"), ("dye-mass", "conservative"),
                         ("dye2-mass", "conservative")):
            pc.register_carray(pc.get_carray_size(), f, "double")
            pc[f][:] = torch.arange(pc.get_carray_size(), device=gpu) * 0.5
            pc.carray_named_groups[group] = pc.carray_named_groups[group] + [f]
            fields.append(f)
    elif how == "missing":
        pc.carray_named_groups["primitive"] = ["nowhere"]
    elif how == "strided":
        wide = torch.zeros((pc.carrays["density"].numel(), 2), dtype=torch.float64, device=gpu)
        wide[:, 0] = pc.carrays["density"]
        wide[:, 1] = -7.0
        pc.carrays["density"] = wide[:, 0]
    elif how == "wide_map":
        pc.carrays["map"] = pc.carrays["map"].long()
    elif how == "box":
        domain = Box(domain)
    prob.mesh.build_geometry(pc, domain)
    plain.mesh.build_geometry(plain.particles, plain.domain_manager)
    tag, image = pc["tag"].cpu().numpy(), pc["map"].cpu().numpy()
    ghosts = np.nonzero(tag)[0]
    assert ghosts.size and (tag[ghosts] == 1).all()
    assert (pc["type"].cpu().numpy()[ghosts] == 2).all()
    for f in fields:
        v = pc[f].cpu().numpy()
        assert np.array_equal(v[ghosts], v[image[ghosts]]), f
    if how == "strided":
        assert (wide[:, 1] == -7.0).all()
    for f in pc.carray_named_groups["position"] + ["volume", "map"]:
        assert np.array_equal(pc[f].cpu().numpy(), plain.particles[f].cpu().numpy()), f
    for f in ("area", "pair-i", "pair-j"):
        assert np.array_equal(prob.mesh.faces[f].cpu().numpy(), plain.mesh.faces[f].cpu().numpy()), f
