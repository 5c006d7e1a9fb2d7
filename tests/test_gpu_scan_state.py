"""What the single-pass scans keep between launches (a ticket, an epoch, tagged
words) must not carry a call's damage into the next one."""
import ctypes as C

import numpy as np
import pytest

from oracle import weld_ref

pytestmark = pytest.mark.gpu


def _mesh(prg, nv, nt, seed):
    rng = np.random.default_rng(seed)
    v = rng.random((nv, 3), dtype=np.float32)
    v[rng.integers(0, nv, nv // 3)] = v[rng.integers(0, nv, nv // 3)]
    t = rng.integers(0, nv, (nt, 3)).astype(np.int32)
    return prg.Mesh(v, t, np.zeros(3, np.float32), 1.0, nv // 2, nt // 2)


# one tile of the scan (2,048 vertices), a few, and the array's limit
@pytest.mark.parametrize("nv", [2048, 2049, 70000, 1 << 19])
def test_noalloc_weld_whatever_the_array_holds(prg, nv):
    """Calls that overlap on a device race for the fixed array and may leave
    anything in it; a later call on its own finds the right mesh."""
    mesh = _mesh(prg, nv, 5000, nv)
    ov, ot, onleaf, oremoved = weld_ref.weld(mesh.vertices, mesh.triangles, mesh.n_leaf_vertices)
    with prg.Reconstructor(max_depth=5) as g:
        address = prg.lib()._ZN3prg20weld_noalloc_scratchEi
        address.restype = C.c_void_p
        hip = prg.lib()  # (the runtime is among the library's dependencies)
        hip.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
        for byte in (0x01, 0x5A, 0xFF):
            print(f"\n[no-alloc weld of {nv} vertices, the array filled with {byte:#x}]", flush=True)
            assert hip.hipMemset(address(0), byte, 48643328) == 0  # PRG_WELD_NOALLOC_BYTES
            assert hip.hipDeviceSynchronize() == 0
            for _ in range(2):
                wm, removed = g.weld_mesh(mesh, noalloc=True)
                assert removed == oremoved and wm.n_leaf_vertices == onleaf
                assert np.array_equal(wm.vertices.view(np.uint32), ov.view(np.uint32))
                assert np.array_equal(wm.triangles, ot)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("nv", [2048, 2049, 100000])
def test_scan_that_gives_up_is_reported(prg, monkeypatch, noalloc, nv):
    """A tile that stops waiting for the tiles before it (test setting: at
    once) leaves no mesh behind that looks right: the call fails, the caller's
    mesh is as it was, and other contexts are not touched."""
    mesh = _mesh(prg, nv, 3000, nv)
    v0, t0 = mesh.vertices.copy(), mesh.triangles.copy()
    want = weld_ref.weld(mesh.vertices, mesh.triangles, mesh.n_leaf_vertices)
    monkeypatch.setenv("PRG_WELD_SPINS", "0")
    g = prg.Reconstructor(max_depth=5)
    monkeypatch.delenv("PRG_WELD_SPINS")
    h = prg.Reconstructor(max_depth=5)
    for _ in range(2):
        print(f"\n[weld of {nv} vertices that gives up at once, noalloc={noalloc}]", flush=True)
        if nv <= 2048:  # one tile waits for none
            wm, _ = g.weld_mesh(mesh, noalloc=noalloc)
            assert np.array_equal(wm.vertices.view(np.uint32), want[0].view(np.uint32))
        else:
            with pytest.raises(prg.PrgError) as e:
                g.weld_mesh(mesh, noalloc=noalloc)
            assert e.value.status == prg.E_HIP
        assert np.array_equal(mesh.vertices, v0) and np.array_equal(mesh.triangles, t0)
        wm, removed = h.weld_mesh(mesh, noalloc=noalloc)
        assert removed == want[3]
        assert np.array_equal(wm.vertices.view(np.uint32), want[0].view(np.uint32))
        assert np.array_equal(wm.triangles, want[1])
    h.close()
    g.close()
