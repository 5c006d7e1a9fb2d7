"""Welds of meshes whose equal vertices follow each other: runs that start and
end anywhere in a wave of 64, span waves and workgroups, and meet the end of
the array, against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import weld_ref

pytestmark = pytest.mark.gpu


def _check(prg, g, v, seed):
    rng = np.random.default_rng(seed)
    t = rng.integers(0, len(v), (500, 3)).astype(np.int32)
    n_leaf = len(v) // 3
    ov, ot, onleaf, oremoved = weld_ref.weld(v, t, n_leaf)
    for noalloc in (False, True):
        wm, removed = g.weld_mesh(prg.Mesh(v, t, np.zeros(3, np.float32), 1.0, n_leaf, 500), noalloc=noalloc)
        assert removed == oremoved and wm.n_leaf_vertices == onleaf
        assert np.array_equal(wm.vertices.view(np.uint32), ov.view(np.uint32))
        assert np.array_equal(wm.triangles, ot)


@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 257, 2049, 50000])
def test_one_position(prg, n):
    print(f"\n[weld: {n} vertices at one position]", flush=True)
    with prg.Reconstructor(max_depth=5) as g:
        _check(prg, g, np.full((n, 3), 0.25, np.float32), n)


@pytest.mark.parametrize("longest", [2, 3, 63, 64, 65, 300, 5000])
def test_runs(prg, longest):
    print(f"\n[weld: runs of up to {longest} equal vertices]", flush=True)
    rng = np.random.default_rng(longest)
    lengths = rng.integers(1, longest + 1, max(20, 40000 // longest))
    # a third of the runs come back to a position met before; coordinates that
    # differ in one word only, among them -0 and +0
    pos = rng.integers(0, 3, (len(lengths), 3)).astype(np.float32)
    pos[::3] = rng.random((len(pos[::3]), 3), dtype=np.float32)
    pos[1::7] *= np.float32(-1.0)
    with prg.Reconstructor(max_depth=5) as g:
        _check(prg, g, np.repeat(pos, lengths, axis=0), longest)
