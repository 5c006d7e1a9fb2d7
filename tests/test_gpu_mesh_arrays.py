"""Who owns the arrays of the Python meshes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("nv,distinct", [(1, 1), (3, 1), (5000, 4999), (300000, 1000), (4000, 4000), (4000, 2000), (4001, 2000)])
def test_welded_mesh_keeps_few_merged_vertices(prg, noalloc, nv, distinct):
    rng = np.random.default_rng(nv)
    pool = rng.random((distinct, 3), dtype=np.float32)
    pick = np.concatenate([np.arange(distinct), rng.integers(0, distinct, nv - distinct)])
    t = rng.integers(0, nv, (20, 3)).astype(np.int32)
    with prg.Reconstructor(max_depth=5) as g:
        print(f"\n[weld {nv} vertices of {distinct} positions, noalloc={noalloc}]", flush=True)
        wm, removed = g.weld_mesh(prg.Mesh(pool[pick], t, np.zeros(3, np.float32), 1.0, nv, 20), noalloc=noalloc)
    assert removed == nv - distinct
    # the array that stays alive with it holds at most twice the mesh's vertices
    assert wm.vertices.shape == (distinct, 3)
    whole = wm.vertices if wm.vertices.base is None else wm.vertices.base
    assert whole.size <= 2 * wm.vertices.size
    assert np.array_equal(wm.vertices.view(np.uint32), pool.view(np.uint32))
    assert np.array_equal(wm.triangles, pick[t])
