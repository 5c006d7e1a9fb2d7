"""A context's buffers share a few allocations: growing them from call to call,
giving parts back and taking them again changes no result, in one context, in
contexts side by side, and for meshes whose arrays outlive the context."""
import threading

import numpy as np
import pytest

import poissonrecon_gpu_amd as prg

pytestmark = pytest.mark.gpu


def _mesh(g, p, q, depth, subdivide=True):
    g.set_max_depth(depth)
    g.set_points(p, q)
    g.build_octree()
    g.compute_divergence()
    g.solve()
    g.isovalue()
    return g.extract_mesh(subdivide)


def _same(a, b):
    assert np.array_equal(a.vertices.view(np.int32), b.vertices.view(np.int32))
    assert np.array_equal(a.triangles, b.triangles)


CLOUDS = [(3000, 6), (40000, 8), (500, 5), (120000, 9), (40000, 8)]


@pytest.fixture(scope="module")
def fresh():
    out = []
    for i, (n, d) in enumerate(CLOUDS):
        p, q = prg.synth_superquadrics(n, seed=10 + i)
        g = prg.Reconstructor(max_depth=d)
        out.append((p, q, d, _mesh(g, p, q, d)))
        g.close()
    return out


@pytest.mark.parametrize("order", [(0, 1, 2, 3, 4), (3, 0, 4, 2, 1)])
def test_one_context_over_sizes(fresh, order):
    g = prg.Reconstructor(max_depth=5)
    for k in order:
        p, q, d, want = fresh[k]
        _same(_mesh(g, p, q, d), want)
        # the weld's arrays come from the same memory and go back to it
        a, ra = g.weld_mesh(want)
        b, rb = g.weld_mesh(want, noalloc=True) if len(want.vertices) <= 100000 else (a, ra)
        assert ra == rb
        _same(a, b)
    g.close()


def test_contexts_side_by_side(fresh):
    bad = []

    def work(order):
        try:
            g = prg.Reconstructor(max_depth=5)
            for k in order:
                p, q, d, want = fresh[k]
                _same(_mesh(g, p, q, d), want)
            g.close()
        except BaseException as e:  # noqa: BLE001 (reported below)
            bad.append(e)

    ts = [threading.Thread(target=work, args=(o,)) for o in [(0, 3, 1), (1, 2, 3), (4, 0, 2)]]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_mesh_outlives_its_context(fresh):
    p, q, d, want = fresh[1]
    g = prg.Reconstructor(max_depth=d)
    m = _mesh(g, p, q, d)
    g.close()
    v, t = m.vertices[5:], m.triangles
    n = len(m.vertices)
    del m
    assert np.array_equal(v, want.vertices[5:]) and np.array_equal(t, want.triangles) and len(v) == n - 5
    v[0] = 0.0  # the arrays are the caller's own
