"""Stages at the sizes where their launch changes: the CFL minimum on both sides
of the line between its small and large blocks."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 255), (2, 256), (2, 257), (2, 32767), (2, 32768), (2, 32769),
                                   (3, 255), (3, 257), (3, 65535), (3, 65536), (3, 65537)])
def test_time_step_around_the_block_size(gpu, dim, n):
    from phd import _native as nat
    print("case time step dim %d, %d cells" % (dim, n), flush=True)
    lib, h = nat.flux(), nat.handle()
    rng = np.random.default_rng(n)
    q = [torch.as_tensor(rng.uniform(0.5, 2.0, n), device=gpu) for _ in range(dim + 2)]
    vol = torch.as_tensor(rng.uniform(0.5, 2.0, n) * 1e-6, device=gpu)
    tag = torch.zeros(n, dtype=torch.int8, device=gpu)
    c = nat.Cells()
    c.dim, c.n_cells, c.tag, c.volume = dim, n, tag.data_ptr(), vol.data_ptr()
    for k, t in enumerate(q):
        c.prim[k] = t.data_ptr()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for at in (n - 1, n // 2, 0):            # the smallest bound in each place
        q[dim + 1][at] = 1e6 * (2 + n - at)
        dt, ref = ctypes.c_double(), ctypes.c_double()
        nat.check(lib.phd_compute_time_step(h, ctypes.byref(c), 1.4, 0.3, 1, ctypes.byref(dt)), "dt")
        nat.check(lib.phd_compute_time_step_noalloc(ctypes.byref(c), 1.4, 0.3, 1, stream,
                                                    ctypes.byref(ref)), "noalloc")
        assert dt.value == ref.value and dt.value > 0
        tag[at] = 1                          # a ghost from here on: the next is the smallest
