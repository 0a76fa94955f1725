"""Routes of single stages at the sizes where they change: the CFL reduction
around its block and grid sizes, the update from flux arrays with faces staged
and gathered, and the TESS limiter on staged and gathered neighbours."""
import ctypes

import numpy as np
import pytest
import torch

from parity import assert_bitwise, check_fields
from test_gpu_cell_order import _renumber_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 262144, 262145, 600001])
def test_time_step_sizes(gpu, dim, n):
    from phd import _native as nat
    print("case time step dim %d, %d cells" % (dim, n), flush=True)
    lib, h = nat.flux(), nat.handle()
    rng = np.random.default_rng(n)
    q = [torch.as_tensor(rng.uniform(0.5, 2.0, n), device=gpu) for _ in range(dim + 2)]
    vol = torch.as_tensor(rng.uniform(0.5, 2.0, n) * 1e-6, device=gpu)
    tag = torch.as_tensor((rng.random(n) < 0.3).astype(np.int8), device=gpu)
    tag[n // 2] = 0
    c = nat.Cells()
    c.dim, c.n_cells, c.tag, c.volume = dim, n, tag.data_ptr(), vol.data_ptr()
    for k, t in enumerate(q):
        c.prim[k] = t.data_ptr()
    for at in (0, n // 2, n - 1):            # the smallest bound in each place
        tag[at] = 0
        q[dim + 1][at] = 1e6 * (2 + at)
        dt, ref = ctypes.c_double(), ctypes.c_double()
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        nat.check(lib.phd_compute_time_step(h, ctypes.byref(c), 1.4, 0.3, 1, ctypes.byref(dt)), "dt")
        nat.check(lib.phd_compute_time_step_noalloc(ctypes.byref(c), 1.4, 0.3, 1, stream,
                                                    ctypes.byref(ref)), "noalloc")
        assert dt.value == ref.value and dt.value > 0


@pytest.mark.parametrize("order", ["builder", "random"])
@pytest.mark.parametrize("name,n", [("sod_2d", 5), ("kh_2d", 41), ("sedov_3d", 7), ("sedov_3d", 15)])
def test_update_from_fluxes_and_tess(gpu, name, n, order):
    """Updated conserved fields and TESS-limited gradients of a random state
    against the oracle, bit for bit."""
    from oracle import oracle
    from phd import problems
    print("case %s n=%d %s" % (name, n, order), flush=True)
    p = problems.PROBLEMS[name](n=n, seed=2)
    pc, mesh = p.particles, p.mesh
    if order == "random":
        _renumber_cells(p, seed=4)
    dim = p.dim
    rng = np.random.default_rng(n)
    for q, f in enumerate(pc.carray_named_groups["primitive"]):
        v = rng.uniform(0.5, 2.0, pc.get_carray_size())
        pc[f][:] = torch.as_tensor(v if q in (0, dim + 1) else v - 1.2, device=gpu)
    p.eos.conservative_from_primitive(pc)
    a = problems.host_arrays(p)
    real = a["tag"] == 0
    p.recon.slope_limiter = 1                        # TESS
    p.recon.compute_gradients(pc, mesh, p.domain_manager)
    grad, rc, _ = oracle.compute_gradients(a, 1)
    assert rc == 0
    got = p.recon.grad.rows().cpu().numpy()
    for q in range(len(grad)):
        assert_bitwise(got[real, q], grad[q][real], "grad %d" % q)
    flux = [rng.normal(0, 1, a["nf"]) for _ in range(dim + 2)]
    p.riemann.fluxes.resize(a["nf"])
    for t, v in zip(p.riemann.fluxes.group("conservative"), flux):
        t[:] = torch.as_tensor(v, device=gpu)
    dt = 1e-4 * float(a["volume"][real].min()) / float(a["area"].max())
    mesh.update_from_fluxes(pc, p.riemann, dt)
    cons, rc, _ = oracle.update_from_fluxes(a, flux, dt)
    assert rc == 0
    check_fields([t.cpu().numpy() for t in pc.group("conservative")], cons, "cons", mask=real,
                 bitwise=True)
