"""Host-side calls in front of the kernels, without a GPU: what the cells view
refuses."""
import pytest

import phd
from phd.views import cells_view


def test_cells_view_refuses_more_fields_than_it_holds():
    pc = phd.HydroParticleCreator(num=4, dim=3, device="cpu")
    c = cells_view(pc)
    assert c.n_cells == 4 and c.prim[4] == pc["pressure"].data_ptr()
    pc.register_carray(4, "dye", "double")
    pc.carray_named_groups["primitive"] = pc.carray_named_groups["primitive"] + ["dye"]
    with pytest.raises(IndexError):
        cells_view(pc)
