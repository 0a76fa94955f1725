"""Which operands the gradient sums take with the Shared arithmetic, on the CPU.

Coordinates, primitives, areas and volumes are checked one by one, and one value
outside sends a whole window of cells to the operators.  Meshes in any unit of
length, fields in any units and velocities that decay ahead of a front have to be
inside; and everything inside gives the operators' bits, up to the limits."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from test_quotients_cpu import lib as quotients   # noqa: F401  (fixture)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "phd-code_amd", "phd", "csrc")
SRC = os.path.join(ROOT, "tests", "quotients", "ranges_host.cpp")
LIB = os.path.join(ROOT, "tests", "quotients", "libranges_host.so")
DEPS = [SRC, os.path.join(CSRC, "quot_dev.h")]
COORD, PRIM, AREA, VOL = range(4)
# the limits that quot_dev.h works out (powers of two)
LIMITS = {COORD: (-100, 150), PRIM: (-240, 150), AREA: (-200, 150), VOL: (-200, 150)}


@pytest.fixture(scope="module")
def ranges():
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(os.path.getmtime(d) for d in DEPS):
        subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-ffp-contract=off",
                        "--offload-arch=gfx950", "-fPIC", "-shared", "-I" + CSRC, "-x", "hip", SRC,
                        "-o", LIB], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    lib = ctypes.CDLL(LIB)
    lib.rh_ok.argtypes = [ctypes.c_int, ctypes.c_double]
    return lib


@pytest.mark.parametrize("length", [1e-12, 1e-6, 1.0, 1e5, 7e10, 1.5e13, 1e15])
@pytest.mark.parametrize("dim", [2, 3])
def test_meshes_in_any_unit_of_length(ranges, dim, length):
    """Cells of this size, with faces down to the smallest that the builder
    keeps (1e-14 of the cell in 2D, 1e-20 of its square in 3D)."""
    assert ranges.rh_ok(COORD, length) and ranges.rh_ok(COORD, 1e6 * length)
    assert ranges.rh_ok(AREA, length ** (dim - 1)) and ranges.rh_ok(VOL, length ** dim)
    assert ranges.rh_ok(AREA, 1e-14 * length if dim == 2 else 1e-20 * length ** 2)


@pytest.mark.parametrize("value", [0.0, -0.0, 1e-31, 1e-40, -1e-60, 1e-70, 1e35, -1e44])
def test_primitives_small_and_large(ranges, value):
    assert ranges.rh_ok(PRIM, value)


@pytest.mark.parametrize("kind", [COORD, PRIM, AREA, VOL])
def test_the_limits(ranges, kind):
    lo, hi = LIMITS[kind]
    assert ranges.rh_ok(kind, 2.0 ** lo) and ranges.rh_ok(kind, 2.0 ** hi)
    assert not ranges.rh_ok(kind, np.nextafter(2.0 ** lo, 0.0))
    assert not ranges.rh_ok(kind, np.nextafter(2.0 ** hi, np.inf))
    for bad in (np.nan, np.inf, -np.inf, 5e-324):
        assert not ranges.rh_ok(kind, bad)
    assert bool(ranges.rh_ok(kind, 0.0)) == (kind != VOL)
    assert bool(ranges.rh_ok(kind, -1.0)) == (kind != VOL)


def _draw(rng, kind, where):
    """A value of the kind's range: near its lower or upper limit, or anywhere."""
    lo, hi = LIMITS[kind]
    e = {"low": lo + rng.integers(0, 3), "high": hi - 1 - rng.integers(0, 3),
         "any": rng.integers(lo, hi)}[where]
    v = rng.uniform(1.0, 2.0) * 2.0 ** int(e)
    return v if kind in (AREA, VOL) or rng.random() < 0.5 else -v


@pytest.mark.parametrize("seed", range(6))
def test_summand_bits_up_to_the_limits(ranges, seed):
    rng = np.random.default_rng(seed)
    kinds = (COORD, COORD, COORD, PRIM, PRIM, AREA, VOL)
    out = np.zeros(2)
    for _ in range(20000):
        where = [("low", "high", "any")[rng.integers(3)] for _ in range(3)]
        at = {COORD: where[0], PRIM: where[1], AREA: where[2], VOL: rng.choice(["low", "high", "any"])}
        v = np.array([_draw(rng, k, at[k]) for k in kinds])
        if rng.random() < 0.3:           # cancellation to the last place
            v[1] = np.nextafter(v[0], 0.0 if abs(v[0]) > 2.0 ** -100 else np.inf * np.sign(v[0]))
        if rng.random() < 0.3:
            v[4] = np.nextafter(v[3], 0.0 if abs(v[3]) > 2.0 ** -240 else np.inf * np.sign(v[3]))
        if rng.random() < 0.1:
            v[rng.integers(0, 6)] = 0.0
        assert all(ranges.rh_ok(k, x) for k, x in zip(kinds, v))
        if ranges.rh_summand(ctypes.c_void_p(v.ctypes.data), ctypes.c_void_p(out.ctypes.data)):
            assert out[:1].view(np.int64) == out[1:].view(np.int64), (v, out)


@pytest.mark.parametrize("dim", [2, 3])
def test_reverse_bits_up_to_the_limits(quotients, dim):   # noqa: F811
    """The gradient's reverse with every operand near a limit, and adjoints near
    theirs (2^+-300), with and without Shared."""
    rng = np.random.default_rng(dim)
    p = lambda a: ctypes.c_void_p(a.ctypes.data)          # noqa: E731
    q = dim + 2
    for trial in range(600):
        deg = int(rng.integers(1, 9))
        where = {k: ("low", "high", "any")[rng.integers(3)] for k in LIMITS}
        put = lambda k, *s: np.array([_draw(rng, k, where[k])    # noqa: E731
                                      for _ in range(int(np.prod(s)))]).reshape(s)
        rows = np.concatenate([put(COORD, deg, dim), put(PRIM, deg, 8 - dim)], axis=1)
        com, area, vol = put(COORD, deg, 3), put(AREA, deg), float(put(VOL, 1)[0])
        pv, xi, cx = put(PRIM, q), put(COORD, 3), put(COORD, 3)
        lgrad = rng.normal(0, 1, dim * q) * 2.0 ** rng.choice([-302, -299, 0, 298, 301])
        got = []
        for fast in (0, 1):
            lself, lnb = np.ones(q), np.zeros(deg * q)
            quotients.qh_grad_vjp(dim, deg, p(rows), p(com), p(area), p(pv), p(xi), p(cx),
                                  ctypes.c_double(vol), p(lgrad), fast, p(lself), p(lnb))
            got.append(np.concatenate([lself, lnb]))
        a, b = got
        same = (a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (trial, where, np.nonzero(~same)[0][:4])
