"""Batched problems whose cells are numbered by rows or at random (the union then
keeps no halos), as in test_gpu_ensemble: every step equal to the per-problem
steps, bit for bit, and the same under every schedule of the gradient kernel."""
import numpy as np
import pytest
import torch

from test_gpu_ensemble import test_ragged_and_single_problem_batches as _check

pytestmark = pytest.mark.gpu


def _order(monkeypatch, how):
    from phd import ensemble
    lattice = ensemble.jittered_lattice

    def ordered(side, dim, seed):
        x = lattice(side, dim, seed, order="rows")
        at = np.random.default_rng(seed).permutation(x[0].size) if how == "shuffled" else slice(None)
        return [np.ascontiguousarray(v[at]) for v in x]
    monkeypatch.setattr(ensemble, "jittered_lattice", ordered)


@pytest.mark.parametrize("how", ["rows", "shuffled"])
@pytest.mark.parametrize("sides", [[150, 5, 120, 90], [200]])
def test_batches_of_scattered_cells(gpu, monkeypatch, sides, how):
    _order(monkeypatch, how)
    print("case batch %s %s" % (sides, how), flush=True)
    _check(gpu, sides)


def test_schedules_on_scattered_cells(gpu, monkeypatch):
    from phd import ensemble as E
    _order(monkeypatch, "shuffled")
    spec = E.draw_problems(3, seed=23)
    spec["side"] = np.array([90, 7, 120], dtype=np.int64)
    ens = E.Ensemble(E.HostEnsemble(spec, n_workers=4), hist_steps=8)
    ens.reset()
    start = ens.state()
    ens.run(3)
    ref = ens.state()
    for block in (64, 128, 256):
        for xcd in (0, 1):
            print("case schedule %d %d" % (block, xcd), flush=True)
            ens.restart(start)
            ens.set_schedule(block, 256, 256, xcd)
            ens.run(3)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(ens.state(), ref)), (block, xcd)
    ens.close()
