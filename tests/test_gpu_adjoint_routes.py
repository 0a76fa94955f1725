"""The gradient's reverse on numberings and values that its staging and its fast
quotients treat differently.

Against the oracle's forward mode, as in test_gpu_adjoint: generators in random
order (most neighbours are not staged; in 2D no halo is kept) and row by row, on
both sides of the line below which a mesh is spread field by field.

With the operators alone: one face of an area below the fast range sends every
cell of its mesh to / and sqrt, and everywhere outside that face's surroundings
the reverse step must keep its bits, on ordinary fields and on fields with values
past the range in some windows."""
import numpy as np
import pytest
import torch

from test_gpu_adjoint import test_rollout_against_forward_mode_ad_of_the_oracle as _check

pytestmark = pytest.mark.gpu


def _order(monkeypatch, how):
    from phd import problems
    lattice = problems.jittered_lattice

    def ordered(n, dim, seed=0, order=None):
        x = lattice(n, dim, seed, order="rows" if how == "rows" else "morton")
        at = np.random.default_rng(7).permutation(x[0].size) if how == "shuffled" else slice(None)
        return [np.ascontiguousarray(v[at]) for v in x]
    monkeypatch.setattr(problems, "jittered_lattice", ordered)


@pytest.mark.parametrize("name,n,pressure", [("kh_2d", 515, None), ("sedov_3d", 63, 1.0)])
def test_reverse_of_large_meshes(gpu, name, n, pressure):
    """Past 1024 windows, where the contributions are combined in blocks of 256."""
    _check(gpu, name, n, pressure, 1, 1, None)


@pytest.mark.parametrize("how", ["rows", "shuffled"])
@pytest.mark.parametrize("name,n,pressure", [("kh_2d", 40, None), ("kh_2d", 185, None),
                                             ("sedov_3d", 12, 1.0), ("sedov_3d", 27, 1.0)])
def test_reverse_on_other_numberings(gpu, monkeypatch, name, n, pressure, how):
    print("case reverse %s n=%d %s" % (name, n, how), flush=True)
    _order(monkeypatch, how)
    _check(gpu, name, n, pressure, 2, 1, None)


def _reverse(gpu, name, n, scale, tiny_face):
    """lambda before one step, for a fixed one after it; and where it is
    compared: cells away from the face nearest the corner."""
    from phd import adjoint, problems
    p = problems.PROBLEMS[name](n=n, seed=3)
    pc, mesh, dim = p.particles, p.mesh, p.dim
    rng = np.random.default_rng(scale)
    na = pc.get_carray_size()
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, na) if q in (0, dim + 1) else rng.normal(0, 0.3, na)
        if 0 < q < dim + 1 and scale:
            some = rng.random(na) < 0.002
            v[some] *= 2.0 ** -rng.integers(0, scale, some.sum())
            v[rng.random(na) < 0.05] = 0.0
        pc[f][:] = torch.as_tensor(v, device=gpu)
    p.domain_manager.update_ghost_fields(pc, pc.carray_named_groups["primitive"], True)
    p.eos.conservative_from_primitive(pc)
    com = np.stack([mesh.faces[f].cpu().numpy() for f in mesh.faces.carray_named_groups["com"]])
    face = int(np.argmin((com ** 2).sum(0)))
    if tiny_face:
        mesh.faces["area"][face] = 1e-70
        mesh.invalidate_plan()
    st = adjoint.StaticStepper(p)
    st.refresh()
    rec, before = st.new_rec(), st.state()
    dt = 0.2 * st.time_step()
    st.step(dt, rec=rec)
    st.set_state(before)
    st.refresh()
    lam = [torch.as_tensor(rng.normal(0, 1, na), device=gpu) for _ in range(dim + 2)]
    out = st.vjp(dt, lam, rec=rec)
    got = [t.cpu().numpy() for t in out]
    x = np.stack([pc[f].cpu().numpy() for f in pc.carray_named_groups["position"]])
    away = np.abs(x - com[:, face:face + 1])
    if name == "kh_2d":                    # periodic
        away = np.minimum(away, 1.0 - away)
    far = (away.max(0) > 10.0 / n) & (pc["tag"].cpu().numpy() == 0)
    st.close()
    return dt, got, far


@pytest.mark.parametrize("scale", [0, 300])
@pytest.mark.parametrize("name,n", [("kh_2d", 60), ("kh_2d", 190), ("sedov_3d", 13), ("sedov_3d", 27)])
def test_reverse_bits_without_fast_quotients(gpu, name, n, scale):
    print("case reverse with operators %s n=%d 2^-%d" % (name, n, scale), flush=True)
    dt, fast, far = _reverse(gpu, name, n, scale, False)
    dt2, slow, _ = _reverse(gpu, name, n, scale, True)
    assert dt == dt2 and far.mean() > 0.05
    for q, (a, b) in enumerate(zip(fast, slow)):
        a, b = a[far], b[far]
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert (a.view(np.int64) == b.view(np.int64)).all(), (q, int((a != b).sum()))
