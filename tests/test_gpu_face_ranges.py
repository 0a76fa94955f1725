"""GPU check of the fused face kernel's fluxes against the materialised states and
the stand-alone solver, bit for bit, for magnitudes up to and past the limits
2^+-132 of the fast quotients (as in test_gpu_quotients)."""
import pytest

from test_gpu_quotients import test_fused_fluxes_equal_materialised as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [120, 131, 136])
@pytest.mark.parametrize("dim,n", [(2, 37), (3, 9)])
def test_fluxes_up_to_the_limits(gpu, dim, n, scale):
    _check(gpu, dim, n, scale)
