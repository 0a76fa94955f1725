"""Host-side calls in front of the kernels, without a GPU: what the cells view
refuses, and that a library handle is refused where torch refuses the GPU."""
import pytest
import torch

import phd
from phd import _native as nat
from phd.views import cells_view


def test_cells_view_refuses_more_fields_than_it_holds():
    pc = phd.HydroParticleCreator(num=4, dim=3, device="cpu")
    c = cells_view(pc)
    assert c.n_cells == 4 and c.prim[4] == pc["pressure"].data_ptr()
    pc.register_carray(4, "dye", "double")
    pc.carray_named_groups["primitive"] = pc.carray_named_groups["primitive"] + ["dye"]
    with pytest.raises(IndexError):
        cells_view(pc)


class _Library(object):
    def __init__(self):
        self.streams = []

    def phd_set_stream(self, h, stream):
        self.streams.append((h, stream))


@pytest.mark.parametrize("device", [None, 0])
def test_handle_refused_in_a_forked_child(monkeypatch, device):
    """A forked child inherits the parent's handles; torch refuses the GPU
    there, and so must the handle, before any call into the library."""
    lib = _Library()
    monkeypatch.setattr(nat, "flux", lambda: lib)
    monkeypatch.setattr(nat, "_handles", {0: 5})

    def refuse(*args):
        raise RuntimeError("Cannot re-initialize CUDA in forked subprocess")
    monkeypatch.setattr(torch.cuda, "current_device", refuse)
    monkeypatch.setattr(torch.cuda, "init", refuse)
    with pytest.raises(RuntimeError, match="forked subprocess"):
        nat.handle(device)
    assert not lib.streams
