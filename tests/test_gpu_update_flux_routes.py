"""The update from flux arrays on both sides of the line from which it leaves the
plain walk of the lists (700 windows of 256 cells in 2D and 256 in 3D with faces in
owner order, 450 and 200 otherwise), against the oracle, bit for bit: cells along
the builder's curve; generators in random order (faces still in owner order, so
that a window's cells have far neighbours and a face named by two windows is
staged in one and gathered in the other); cells renumbered after the faces; and
faces renumbered (no owner order: the sliced lists).  Some windows own more faces
than are staged.  The fault it reports is the oracle's first."""
import numpy as np
import pytest
import torch

from parity import check_fields
from test_gpu_cell_order import _renumber_cells
from test_gpu_face_order import _owner_runs, _renumber

pytestmark = pytest.mark.gpu

# windows from which the walk is left, with faces in owner order or not
MIN_WINDOWS = {(2, True): 700, (3, True): 256, (2, False): 450, (3, False): 200}
CASES = [(name, n, above, order) for name, n, above in
         (("kh_2d", 410, False), ("kh_2d", 430, True), ("sedov_3d", 36, False), ("sedov_3d", 42, True))
         for order in ("builder", "shuffled", "cells")] + \
        [("kh_2d", 330, False, "faces"), ("kh_2d", 345, True, "faces"),
         ("sedov_3d", 33, False, "faces"), ("sedov_3d", 37, True, "faces")]


@pytest.mark.parametrize("name,n,above,order", CASES)
def test_update_from_fluxes_both_sides(gpu, monkeypatch, name, n, above, order):
    from oracle import oracle
    from phd import problems
    print("case %s n=%d %s" % (name, n, order), flush=True)
    if order == "shuffled":
        lattice = problems.jittered_lattice

        def shuffled(*args, **kw):
            x = lattice(*args, **kw)
            perm = np.random.default_rng(7).permutation(x[0].size)
            return [np.ascontiguousarray(v[perm]) for v in x]
        monkeypatch.setattr(problems, "jittered_lattice", shuffled)
    p = problems.PROBLEMS[name](n=n, seed=2)
    pc, mesh, dim = p.particles, p.mesh, p.dim
    if order == "cells":
        _renumber_cells(p, seed=4)
    if order == "faces":
        _renumber(p, seed=11)
    windows = (pc.get_carray_size() + 255) // 256
    assert (windows >= MIN_WINDOWS[dim, order != "faces"]) == above, windows
    rng = np.random.default_rng(n)
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, pc.get_carray_size())
        pc[f][:] = torch.as_tensor(v if q in (0, dim + 1) else v - 1.2, device=gpu)
    p.eos.conservative_from_primitive(pc)
    a = problems.host_arrays(p)
    real = a["tag"] == 0
    assert _owner_runs(a) == (order != "faces")
    if order in ("builder", "shuffled"):     # windows own more than is staged (800, 1750)
        assert (np.diff(a["pair_i"]) >= 0).all()
        assert np.bincount(a["pair_i"] // 256).max() > (800 if dim == 2 else 1750)
    flux = [rng.normal(0, 1, a["nf"]) for _ in range(dim + 2)]
    p.riemann.fluxes.resize(a["nf"])
    arrays = p.riemann.fluxes.group("conservative")
    for t, v in zip(arrays, flux):
        t[:] = torch.as_tensor(v, device=gpu)
    dt = 1e-4 * float(a["volume"][real].min()) / float(a["area"].max())
    mesh.update_from_fluxes(pc, p.riemann, dt)
    cons, rc, _ = oracle.update_from_fluxes(a, flux, dt)
    assert rc == 0
    check_fields([t.cpu().numpy() for t in pc.group("conservative")], cons, "cons", mask=real,
                 bitwise=True)

    # two faults: an energy in the middle of the list, a mass after it
    a = problems.host_arrays(p)
    flux = [np.zeros(a["nf"]) for _ in range(dim + 2)]
    at, later = a["nf"] // 2, (9 * a["nf"]) // 10
    while not (real[a["pair_i"][at]] and real[a["pair_j"][at]]):
        at += 1
    while not (real[a["pair_i"][later]] and real[a["pair_j"][later]]):
        later += 1
    flux[dim + 1][at] = 1e6 / a["area"][at]
    flux[0][later] = 1e6 / a["area"][later]
    _, rc, bad = oracle.update_from_fluxes(a, flux, 1.0)
    assert rc == 3 and bad == at
    for t, v in zip(arrays, flux):
        t[:] = torch.as_tensor(v, device=gpu)
    with pytest.raises(RuntimeError, match="Energy less than zero in flux update") as e:
        mesh.update_from_fluxes(pc, p.riemann, 1.0)
    assert e.value.index == bad
