"""Sizes at the edges of the kernels' tiles, bit for bit against the oracles:
octrees around the look-back scans' and the sort's tile sizes, clouds of many
points per leaf cell (the dense vector-field tiles and the path beyond them),
and welds around the table pass's tile size."""
import numpy as np
import pytest

import oracle as orc
from oracle import weld_ref

pytestmark = pytest.mark.gpu

BUFS_OCTREE = ["BUF_POINTS", "BUF_NORMALS", "BUF_POINT_LEAF", "BUF_KEY", "BUF_PIDX", "BUF_PNUM", "BUF_PARENT",
               "BUF_CHILDREN", "BUF_DIDX", "BUF_DNUM", "BUF_NEIGHS"]


def _both(prg, p, q, depth):
    o = orc.Oracle(depth)
    o.set_points(p, q)
    o.build_octree()
    g = prg.Reconstructor(max_depth=depth)
    g.set_points(p, q)
    g.build_octree()
    return g, o


@pytest.mark.parametrize("n,depth,places", [(2, 4, 0), (255, 6, 0), (256, 6, 0), (257, 6, 0), (2047, 7, 0),
                                            (2048, 7, 0), (2049, 7, 0), (4095, 8, 0), (4096, 8, 0), (4097, 8, 0),
                                            (65536, 8, 0), (65537, 9, 0), (5000, 7, 40), (70000, 9, 3000)])
def test_octree_at_tile_edges(prg, n, depth, places):
    print(f"\n[octree: {n} points at depth {depth}, {places} places]", flush=True)
    p, q = prg.synth_torus(n, n)
    if places:  # many points of one place
        k = np.random.default_rng(n).integers(0, places, n)
        p, q = p[k], q[k]
    g, o = _both(prg, p, q, depth)
    assert g.level_info()[0].tolist() == o.level_info()[0].tolist()
    for b in BUFS_OCTREE:
        a, r = g.read_buffer(getattr(prg, b)), o.read_buffer(getattr(prg, b))
        assert a.shape == r.shape and np.array_equal(a.view(np.uint32), r.view(np.uint32)), b
    g.close()
    o.close()


@pytest.mark.parametrize("n,depth", [(30000, 5), (30000, 6), (60000, 7), (200000, 8)])
def test_dense_vector_field(prg, n, depth):
    print(f"\n[vector field: {n} points at depth {depth}]", flush=True)
    p, q = prg.synth_sphere(n, 5)
    g, o = _both(prg, p, q, depth)
    g.compute_divergence()
    o.compute_divergence()
    a, r = g.read_buffer(prg.BUF_VECTOR_FIELD), o.read_buffer(prg.BUF_VECTOR_FIELD)
    assert np.array_equal(a.view(np.uint32), r.view(np.uint32))
    g.close()
    o.close()


@pytest.mark.parametrize("n,values", [(2, 1), (3, 1), (2047, 700), (2048, 2048), (2049, 5), (4096, 1), (40000, 9000)])
def test_weld_at_tile_edges(prg, n, values):
    rng = np.random.default_rng(n)
    v = rng.standard_normal((values, 3)).astype(np.float32)
    v[:: 3, 0] = np.where(rng.random(len(v[:: 3])) < 0.5, np.float32(-0.0), np.float32(0.0))
    v[1:: 5, 1] = np.nan
    v = v[rng.integers(0, values, n)]
    t = rng.integers(0, n, (3 * n, 3)).astype(np.int32)
    for n_leaf in (0, 1, n // 2, n):
        with prg.Reconstructor(max_depth=4) as g:
            for noalloc in (False, True):
                m, removed = g.weld_mesh(prg.Mesh(v, t, np.zeros(3, np.float32), 1.0, n_leaf, len(t)), noalloc=noalloc)
                ov, ot, onleaf, oremoved = weld_ref.weld(v, t, n_leaf)
                assert removed == oremoved and m.n_leaf_vertices == onleaf
                assert np.array_equal(m.vertices.view(np.uint32), ov.view(np.uint32))
                assert np.array_equal(m.triangles, ot)


@pytest.mark.parametrize("n,depth,refresh", [(900, 6, 1), (3000, 7, 1), (3000, 7, 3), (60000, 7, 2), (20000, 8, 4)])
def test_residual_refresh_on_tiles(prg, n, depth, refresh):
    """Solves that recompute r = b - A x every few iterations, ten iterations on
    both sides (the tolerance of the solve without a refresh)."""
    print(f"\n[refresh: {n} points at depth {depth}, every {refresh}]", flush=True)
    p, q = prg.synth_torus(n, n)
    g, o = _both(prg, p, q, depth)
    g.close()
    o.compute_divergence()
    with prg.Reconstructor(max_depth=depth, cg_fixed_iters=10, cg_refresh=refresh) as g2:
        g2.set_points(p, q)
        g2.build_octree()
        g2.write_buffer(prg.BUF_DIVERGENCE, o.read_buffer(prg.BUF_DIVERGENCE))
        g2.solve()
        xg = g2.read_buffer(prg.BUF_SOLUTION).astype(np.float64)
    o.solve(mode=0, refresh=refresh, fixed_iters=10)
    xo = o.read_buffer(prg.BUF_SOLUTION).astype(np.float64)
    assert np.linalg.norm(xg - xo) <= 1e-5 * np.linalg.norm(xo)
    o.close()
