"""GPU check of the frozen-mesh step on both sides of the line below which the
gradients are formed field by field (128 windows of 256 cells in 2D, 100 in 3D)
against the oracle's step, and of a one-window mesh."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n", [("kh_2d", 10), ("kh_2d", 175), ("kh_2d", 181),
                                    ("sedov_3d", 4), ("sedov_3d", 27), ("sedov_3d", 30)])
def test_both_sides_of_the_field_split(gpu, name, n):
    from oracle import oracle
    from phd import problems
    prob = problems.PROBLEMS[name](n=n, seed=3)
    pc = prob.particles
    real = pc["tag"] == 0
    rng = np.random.default_rng(5)
    for f in pc.carray_named_groups["primitive"]:     # every field with a gradient
        z = torch.as_tensor(rng.uniform(0.0, 0.05, int(real.sum())), device=pc.device)
        pc[f][real] = pc[f][real] * (1 + z) + (0.0 if f in ("density", "pressure") else 1.0) * z
    prob.eos.conservative_from_primitive(pc)
    step = problems.FrozenStep(prob)
    step.prologue()
    dt = step.time_step()
    a = problems.host_arrays(prob)
    ref = oracle.core_step(a, dt)
    assert ref["rc"] == 0
    step.run(dt)
    step.check()
    torch.cuda.synchronize()
    at = a["tag"] == 0
    pairs = list(zip(prob.riemann.fluxes.group("conservative"), ref["flux"])) + \
        [(g[torch.as_tensor(at, device=g.device)], w[at])
         for g, w in zip(pc.group("conservative"), ref["cons"])]
    for got, want in pairs:
        got = got.cpu().numpy()
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
