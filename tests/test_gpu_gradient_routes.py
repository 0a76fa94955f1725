"""The gradient kernel of production sizes (all fields at once, from 128 windows of
256 cells in 2D and 100 in 3D) on cell numberings that its staging treats
differently, against the oracle, bit for bit:

  builder     along the space-filling curve: a window keeps its whole halo
  strips      4 cells wide (2D): a halo past what is staged, kept in part
  rows        one lattice row after the other: no halo in 2D
  shuffled    generators in random order, faces in owner order: no halo in 2D
  renumbered  random order given after the faces': no halo in 2D

and on fields in and past the ranges of the fast quotients, in cells spread over
the windows and so also among the neighbours that are not staged."""
import numpy as np
import pytest
import torch

from parity import assert_bitwise, check_fields
from test_gpu_cell_order import _renumber_cells

pytestmark = pytest.mark.gpu

CASES = [(name, n, order) for name, n in (("kh_2d", 185), ("sedov_3d", 30))
         for order in ("builder", "strips", "rows", "shuffled", "renumbered")
         if order != "strips" or name == "kh_2d"]


def _reorder(problems, monkeypatch, order):
    """Let the set-ups draw their generators in another order."""
    lattice = problems.jittered_lattice

    def ordered(m, dim, seed):
        x = lattice(m, dim, seed, order="rows")
        at = np.arange(x[0].size)
        if order == "shuffled":
            at = np.random.default_rng(7).permutation(at.size)
        elif order == "strips":
            i, j = [np.clip((v * m).astype(int), 0, m - 1) for v in x]
            at = np.lexsort((i, j, i // 4))
        return [np.ascontiguousarray(v[at]) for v in x]
    monkeypatch.setattr(problems, "jittered_lattice",
                        lambda m, dim, seed=0, order=None: ordered(m, dim, seed))


def _problem(problems, monkeypatch, name, n, order):
    if order in ("rows", "strips", "shuffled"):
        _reorder(problems, monkeypatch, order)
    p = problems.PROBLEMS[name](n=n, seed=1)
    if order == "renumbered":
        _renumber_cells(p, seed=4)
    assert p.particles.get_carray_size() // 256 >= (128 if p.dim == 2 else 100)
    return p


def _outside(a):
    """Share of the real cells' list entries that leave their window, and the
    distinct outside cells of window 20."""
    f = a["nbr_face"][:a["nbr_off"][-1]]
    cell = np.repeat(np.arange(a["n"]), np.diff(a["nbr_off"]))
    other = np.where(a["pair_i"][f] == cell, a["pair_j"][f], a["pair_i"][f])
    real = a["tag"][cell] == 0
    out = real & (cell // 256 != other // 256)
    return out.sum() / real.sum(), np.unique(other[out & (cell // 256 == 20)]).size


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("scale", [0, 130, 285, 330])
@pytest.mark.parametrize("name,n,order", CASES)
def test_gradients_over_orders_and_scales(gpu, monkeypatch, name, n, order, scale, limiter):
    from oracle import oracle
    from phd import problems
    print("case gradients %s n=%d %s 2^+-%d limiter %d" % (name, n, order, scale, limiter), flush=True)
    p = _problem(problems, monkeypatch, name, n, order)
    pc = p.particles
    na = pc.get_carray_size()
    rng = np.random.default_rng(scale + n)
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, na) if q in (0, p.dim + 1) else rng.normal(0, 1, na)
        some = rng.random(na) < 0.002
        v[some] *= 2.0 ** rng.integers(-scale, min(scale, 190) + 1, some.sum())
        v[rng.random(na) < 0.05] = 0.0
        pc[f][:] = torch.as_tensor(v, device=gpu)
    a = problems.host_arrays(p)
    if p.dim == 2 and scale == 0:
        share, halo = _outside(a)
        assert (share > 0.25) == (order in ("rows", "shuffled", "renumbered"))
        if share < 0.25:
            assert (halo > 112) == (order == "strips")
    p.recon.slope_limiter = limiter
    p.recon.compute_gradients(pc, p.mesh, p.domain_manager)
    grad, rc, _ = oracle.compute_gradients(a, limiter)
    assert rc == 0
    real = a["tag"] == 0
    got = p.recon.grad.rows().cpu().numpy()
    for q in range(len(grad)):
        assert_bitwise(got[real, q], grad[q][real], "grad %d" % q)


@pytest.mark.parametrize("name,n,order", CASES)
def test_core_step_over_orders(gpu, monkeypatch, name, n, order):
    """Gradients bit for bit; fluxes and updated conserved fields to the parity
    bound (the two-rarefaction powers need not give the same bits)."""
    from oracle import oracle
    from phd import problems
    print("case step %s n=%d %s" % (name, n, order), flush=True)
    p = _problem(problems, monkeypatch, name, n, order)
    pc = p.particles
    rng = np.random.default_rng(n)
    for f in pc.carray_named_groups["primitive"]:
        z = torch.as_tensor(rng.uniform(0.0, 0.05, pc.get_carray_size()), device=gpu)
        pc[f][:] = pc[f] * (1 + z) + (0.0 if f in ("density", "pressure") else 1.0) * z
    p.domain_manager.update_ghost_fields(pc, pc.carray_named_groups["primitive"])
    p.eos.conservative_from_primitive(pc)
    step = problems.FrozenStep(p)
    step.prologue()
    dt = step.time_step()
    a = problems.host_arrays(p)
    ref = oracle.core_step(a, dt, solver=step.solver, boost=bool(step.boost),
                           gizmo=bool(step.gizmo), limiter=step.limiter)
    assert ref["rc"] == 0 and ref["bad"] < 0
    step.run(dt)
    step.check()
    torch.cuda.synchronize()
    real = a["tag"] == 0
    rows = p.recon.grad.rows().cpu().numpy()
    check_fields([rows[:, q] for q in range(len(ref["grad"]))], ref["grad"], "grad", mask=real,
                 bitwise=True)
    check_fields([t.cpu().numpy() for t in p.riemann.fluxes.group("conservative")], ref["flux"], "flux")
    check_fields([t.cpu().numpy() for t in pc.group("conservative")], ref["cons"], "cons", mask=real)
