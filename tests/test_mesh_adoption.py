"""The Python meshes take over arrays that the library allocated: each has one
owner at every step, also when taking over fails half-way."""
import ctypes as C
import gc

import numpy as np
import pytest

_libc = C.CDLL(None)
_libc.malloc.restype = C.c_void_p
_libc.malloc.argtypes = [C.c_size_t]


def _mesh(prg, nv, nt):
    m = prg.PrgMesh()
    m.n_vertices, m.n_triangles = nv, nt
    m.vertices = C.cast(_libc.malloc(12 * nv + 4), C.POINTER(C.c_float))
    m.triangles = C.cast(_libc.malloc(12 * nt + 4), C.POINTER(C.c_int32))
    for i in range(3 * nv):
        m.vertices[i] = i
    for i in range(3 * nt):
        m.triangles[i] = -i
    return m


@pytest.mark.parametrize("nv,nt", [(0, 0), (4, 2), (1000, 0)])
def test_adopted_arrays(prg, nv, nt):
    m = _mesh(prg, nv, nt)
    v, t = prg._adopt_mesh(m)
    assert not m.vertices and not m.triangles  # nothing left for prg_mesh_release
    prg.lib().prg_mesh_release(C.byref(m))
    gc.collect()
    assert v.shape == (nv, 3) and t.shape == (nt, 3) and v.flags.writeable
    assert np.array_equal(v.ravel(), np.arange(3 * nv, dtype=np.float32))
    assert np.array_equal(t.ravel(), -np.arange(3 * nt, dtype=np.int32))


def test_failure_half_way_leaves_one_owner(prg, monkeypatch):
    owned = []

    class Failing(prg._HostArray):
        def __init__(self, pointer, rows, dtype, **field):
            if "triangles" in field:
                raise MemoryError
            super().__init__(pointer, rows, dtype, **field)
            owned.append(self)

    monkeypatch.setattr(prg, "_HostArray", Failing)
    m = _mesh(prg, 5, 5)
    with pytest.raises(MemoryError):
        prg._adopt_mesh(m)
    assert len(owned) == 1
    assert not m.vertices  # freed by its view alone
    assert m.triangles  # still the mesh's, freed by prg_mesh_release
    prg.lib().prg_mesh_release(C.byref(m))
