"""Which states the face kernels' Shared arithmetic takes, on the CPU: densities
and pressures in any unit (1.8e-40 to 5.4e39), with the operators' bits up to the
limits."""
import numpy as np
import pytest

from test_quotients_cpu import Faces, NF, lib   # noqa: F401  (lib: fixture)


def _scale(F, dim, d, p):
    """Densities times d, pressures times p, their gradients with them, and
    velocities and their gradients by sqrt(p / d)."""
    q = dim + 2
    f = np.array([d] + [np.sqrt(p / d)] * dim + [p])
    for r in (F.ri, F.rj):
        r[:, :q] *= f
        r[:, q:q + dim * q] *= np.repeat(f, dim)
    F.fv *= np.sqrt(p / d)


@pytest.mark.parametrize("d,p", [(1e-31, 1e-31), (1e-30, 1e-18), (1e-38, 1e-38), (1e33, 1e33),
                                 (1e-24, 1e-12), (1e15, 1e35)])
@pytest.mark.parametrize("dim", [2, 3])
def test_states_in_any_unit_are_accepted(lib, dim, d, p):   # noqa: F811
    for hllc in (0, 1):
        for gizmo in (0, 1):
            F = Faces(dim, 21)
            _scale(F, dim, d, p)
            ok, same = F.run(lib, hllc, 1.4, 1e-4 / np.sqrt(p / d), 1, gizmo)
            assert ok.mean() > 0.99, (hllc, gizmo, ok.mean())
            assert same[ok].all()


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("dim", [2, 3])
def test_bits_up_to_the_limits(lib, dim, seed):   # noqa: F811
    """Densities and pressures of each side anywhere up to and just past 2^+-132,
    velocities from 2^-510 to 2^102."""
    seen = 0
    F = Faces(dim, 300 + seed)
    rng, q = F.rng, dim + 2
    for r in (F.ri, F.rj):
        for col in (0, q - 1):
            edge = rng.choice([-132, 131, 0], NF) + rng.integers(-1, 2, NF)
            e = np.where(rng.random(NF) < 0.5, edge, rng.integers(-133, 134, NF))
            r[:, col] = rng.uniform(1.0, 2.0, NF) * 2.0 ** e
        e = rng.choice([-510, -499, -300, -60, 0, 60, 99, 101], (NF, dim))
        r[:, 1:1 + dim] = rng.choice([-1.0, 0.0, 1.0], (NF, dim)) * 2.0 ** e
        r[:, q:-dim] *= 0.0 if seed % 2 else 2.0 ** -120.0
    with np.errstate(all="ignore"):
        for hllc in (0, 1):
            for boost in (0, 1):
                for gamma in (1.4, 1.0 + 2.0 ** -10, 64.0):
                    ok, same = F.run(lib, hllc, gamma, 2.0 ** -40, boost, seed & 1)
                    assert same[ok].all(), (hllc, boost, gamma, np.nonzero(ok & ~same)[0][:5])
                    seen += ok.sum()
    assert seen > 0
