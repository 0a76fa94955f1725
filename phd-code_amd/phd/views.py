"""Builders of the C-ABI views (phd_cells / phd_faces) over containers.

A step builds a dozen of them, so each is packed in one call from the arrays'
pointers (a quarter of the host time of filling the fields one by one); nothing
is kept between calls."""
import struct

from . import _native as nat

# phd_cells: dim, n_cells; tag, type, map, x[3], dcom[3], volume, prim[5],
# cons[5], w[3].  phd_faces: n_faces (padded); area, com[3], normal[3],
# velocity[3], pair_i, pair_j, nbr_off, nbr_face.
_CELLS = struct.Struct("@ii23P")
_FACES = struct.Struct("@i14P")
assert _CELLS.size == nat.ctypes.sizeof(nat.Cells) and _FACES.size == nat.ctypes.sizeof(nat.Faces)


def _ptrs(arrays, names, room):
    p = [arrays[f].data_ptr() for f in names]
    if len(p) > room:
        raise IndexError("a group of %d fields where the view holds %d" % (len(p), room))
    return p + [0] * (room - len(p))


def cells_view(particles):
    """phd_cells over a particle container (reals first, then ghosts)."""
    g, a = particles.carray_named_groups, particles.carrays
    one = [a[f].data_ptr() if f in a else 0 for f in ("map", "volume")]
    return nat.Cells.from_buffer_copy(_CELLS.pack(
        len(g["position"]), particles.get_carray_size(), a["tag"].data_ptr(),
        a["type"].data_ptr(), one[0], *_ptrs(a, g["position"], 3), *_ptrs(a, g.get("dcom", ()), 3),
        one[1], *_ptrs(a, g["primitive"], 5), *_ptrs(a, g["conservative"], 5),
        *_ptrs(a, g.get("w", ()), 3)))


def faces_view(mesh):
    """phd_faces over a mesh's face container and per-cell face lists."""
    faces, nbr = mesh.faces, mesh.neighbors
    g, a = faces.carray_named_groups, faces.carrays
    return nat.Faces.from_buffer_copy(_FACES.pack(
        faces.get_carray_size(), a["area"].data_ptr(), *_ptrs(a, g["com"], 3),
        *_ptrs(a, g["normal"], 3), *_ptrs(a, g["velocity"], 3), a["pair-i"].data_ptr(),
        a["pair-j"].data_ptr(), nbr.offsets.data_ptr(),
        nbr.faces.data_ptr() if nbr.faces.numel() else 0))
