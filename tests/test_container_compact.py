"""CarrayContainer drops tagged items wherever they stand: the kept ones keep
their order and their values, also where nothing has to move."""
import pytest
import torch

import phd


@pytest.mark.parametrize("tags", [[], [1], [0], [1, 1, 0], [0, 1], [1, 0, 1], [0, 0], [0, 1, 1, 0],
                                  [1, 1, 1], [1, 0, 0]])
def test_remove_tagged_keeps_order(tags):
    c = phd.CarrayContainer(len(tags), {"v": "double", "tag": "int"}, device="cpu")
    c["v"][:] = torch.arange(len(tags), dtype=torch.float64)
    c["tag"][:] = torch.tensor(tags, dtype=torch.int8)
    c.remove_tagged_particles(0)
    want = [float(k) for k, t in enumerate(tags) if t != 0]
    assert c["v"].tolist() == want and c.get_carray_size() == len(want)
    assert c["tag"].tolist() == [t for t in tags if t != 0]
