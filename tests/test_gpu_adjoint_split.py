"""GPU check of the gradient's reverse on both sides of the line below which a
mesh is spread over the chip field by field: the rollout's gradient against the
oracle's forward mode, as in test_gpu_adjoint, on meshes of a few windows less
and a few more than 128 (2D) and 80 (3D)."""
import pytest

from test_gpu_adjoint import test_rollout_against_forward_mode_ad_of_the_oracle as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n,pressure", [("kh_2d", 175, None), ("kh_2d", 181, None),
                                             ("sedov_3d", 24, 1.0), ("sedov_3d", 27, 1.0)])
def test_both_sides_of_the_field_split(gpu, name, n, pressure):
    _check(gpu, name, n, pressure, 2, 1, None)
