"""Batched problems whose cells are numbered by rows or at random (the union then
keeps no halos), as in test_gpu_ensemble: every step equal to the per-problem
steps, bit for bit."""
import numpy as np
import pytest

from test_gpu_ensemble import test_ragged_and_single_problem_batches as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["rows", "shuffled"])
@pytest.mark.parametrize("sides", [[150, 5, 120, 90], [200]])
def test_batches_of_scattered_cells(gpu, monkeypatch, sides, how):
    from phd import ensemble
    lattice = ensemble.jittered_lattice

    def ordered(side, dim, seed):
        x = lattice(side, dim, seed, order="rows")
        at = np.random.default_rng(seed).permutation(x[0].size) if how == "shuffled" else slice(None)
        return [np.ascontiguousarray(v[at]) for v in x]
    monkeypatch.setattr(ensemble, "jittered_lattice", ordered)
    print("case batch %s %s" % (sides, how), flush=True)
    _check(gpu, sides)
