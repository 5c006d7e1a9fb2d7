"""The workloads that this library's speed is measured on.

Each case is one pass a user's program makes through the public entry points:
a point cloud to its mesh or to its implicit function, a batch of clouds, the
welding of a mesh, and the warm-start network's inference and training.  Sizes
are those of the tests and of bench.py: 2,000 to 4,000,000 points, octree
depths 4 to 10, networks on 16^3 to 64^3 grids.

`listed()` names the fixed cases, `draw(rng)` gives further ones of the same
ranges, `prepare` makes what a program holds before the call, `run` is one
pass, `work` what the pass cannot do without, and `exact` the outputs in 64
bits where plain numpy or torch gives them.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch  # before the library: one HIP runtime in the process

import poissonrecon_gpu_amd as prg

# Surface area of the generators' shapes after normalisation (the longest
# extent becomes 0.8): sphere of radius 0.4, torus 0.30/0.12 in extent 0.84,
# and about 1 for a union of superquadrics.
AREA = {"sphere": 2.0, "torus": 1.3, "superquadrics": 1.0}

# Channels of the network's 3x3x3 convolutions, in parameter order.
CONVS = [(16, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 64), (64, 64), (128, 64), (64, 64),
         (96, 32), (32, 32), (48, 16), (16, 16)]
LEVEL = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0]  # halvings of the grid at each convolution


def _mesh(name, shape, points, depth, subdivide=True, source="host", sink="host"):
    return {"name": name, "kind": "mesh", "shape": shape, "points": points, "depth": depth, "subdivide": subdivide,
            "source": source, "sink": sink}


def listed():
    return [
        # a preview of a small scan: launches and host work are most of it
        _mesh("mesh_sphere_2k_d5", "sphere", 2000, 5),
        # the reference's own example size (a 36 K-point scan at depth 8), ordinary host memory
        _mesh("mesh_sphere_36k_d8", "sphere", 35947, 8),
        # the leaf-level surface alone, from points that a GPU program already holds
        _mesh("leaf_torus_500k_d9", "torus", 500000, 9, subdivide=False, source="device", sink="pinned"),
        # an ordinary scan from host memory to the whole mesh, buffers kept by the program
        _mesh("mesh_torus_500k_d9", "torus", 500000, 9, source="pinned", sink="pinned"),
        # the headline workload: 2 M points at the deepest octree
        _mesh("mesh_superquadrics_2M_d10", "superquadrics", 2000000, 10, source="pinned", sink="pinned"),
        # few points for their depth: most of the surface lies in coarse leaves
        _mesh("mesh_superquadrics_150k_d10", "superquadrics", 150000, 10, source="pinned", sink="pinned"),
        # the largest clouds of the many-clouds workload
        _mesh("mesh_superquadrics_4M_d10", "superquadrics", 4000000, 10, source="device", sink="pinned"),
        # the implicit function itself (solution, isovalue, values at the samples), no mesh
        {"name": "field_superquadrics_80k_d9", "kind": "field", "shape": "superquadrics", "points": 80000, "depth": 9},
        # many clouds in one call, four worker contexts
        {"name": "batch_6_clouds", "kind": "batch", "clouds": 6, "smallest": 10000, "largest": 1000000},
        # seam vertices of a subdivided mesh merged
        {"name": "weld_300k", "kind": "weld", "vertices": 300000, "triangles": 400000},
        # the learned warm start's network: one prediction, and a training step of bench.py's size
        {"name": "unet_predict_64", "kind": "predict", "grid": 64},
        {"name": "unet_train_64_b8", "kind": "train", "grid": 64, "batch": 8},
    ]


def _usual_depth(n):
    """The many-clouds workload's rule for a cloud's depth, continued to smaller clouds."""
    return max(4, min(10, 7 + round(math.log2(n / 1e4) / 2)))


def draw(rng):
    kind = rng.choices(["mesh", "field", "weld", "predict", "train", "batch"], [12, 2, 2, 1, 1, 1])[0]
    if kind in ("mesh", "field"):
        n = round(math.exp(rng.uniform(math.log(2000), math.log(2.2e6))))
        shape = rng.choice(sorted(AREA))
        d = _usual_depth(n) + rng.choice([-1, 0, 0, 0, 1])
        d = max(4, min(10 if n >= 150000 * AREA[shape] else 9, d))
        c = {"kind": kind, "shape": shape, "points": n, "depth": d}
        if kind == "mesh":
            c.update(subdivide=rng.random() < 0.8, source=rng.choice(["host", "pinned", "device"]),
                     sink=rng.choice(["host", "pinned"]))
        return c
    if kind == "weld":
        n = round(math.exp(rng.uniform(math.log(1000), math.log(1.5e6))))
        return {"kind": kind, "vertices": n, "triangles": round(n * rng.uniform(1.2, 2.0))}
    if kind == "predict":
        return {"kind": kind, "grid": rng.choice([16, 32, 64]), "level": round(rng.uniform(0.2, 0.45), 4)}
    if kind == "train":
        return {"kind": kind, "grid": rng.choice([16, 32]), "batch": rng.randrange(1, 9)}
    lo = round(math.exp(rng.uniform(math.log(3000), math.log(30000))))
    return {"kind": kind, "clouds": rng.randrange(2, 7), "smallest": lo, "largest": round(lo * rng.uniform(8, 30))}


# ---- inputs ---------------------------------------------------------------------------
def _cloud(shape, n, seed):
    if shape == "sphere":
        return prg.synth_sphere(n, seed)
    if shape == "torus":
        return prg.synth_torus(n, seed)
    return prg.synth_superquadrics(n, 3, 0.001, seed)


def _pinned(a):
    t = torch.empty(a.shape, dtype=torch.from_numpy(a).dtype, pin_memory=True)
    t.copy_(torch.from_numpy(a))
    return t


def _batch_sizes(case):
    k, lo, hi = case["clouds"], math.log(case["smallest"]), math.log(case["largest"])
    return [round(math.exp(lo + (hi - lo) * i / (k - 1))) for i in range(k)]


def _planted_mesh(case, seed):
    """A mesh of random vertices, a tenth of which repeat another one."""
    rng = np.random.default_rng(seed)
    n = case["vertices"]
    v = rng.random((n, 3), dtype=np.float32)
    k = n // 10
    order = rng.permutation(n)
    v[order[:k]] = v[order[k + rng.integers(0, n - k, k)]]
    t = rng.integers(0, n, (case["triangles"], 3)).astype(np.int32)
    return v, t, n // 2


def _num_params():
    return sum(27 * i * o + o for i, o in CONVS) + 17


def _net_params(seed):
    """He-normal convolutions with small biases, in the library's flat layout."""
    rng = np.random.default_rng(1000 + seed)
    p = []
    for i, o in CONVS:
        p.append(rng.standard_normal(27 * o * i) * math.sqrt(2.0 / (27 * i)))
        p.append(rng.standard_normal(o) * 0.02)
    p.append(rng.standard_normal(16) * 0.25)
    p.append(np.zeros(1))
    return np.concatenate(p).astype(np.float32)


def _samples(case, seed):
    """Divergence, node mask and solution grids: values on the cells near a
    sphere's surface, as an octree's depth holds them."""
    rng = np.random.default_rng(seed)
    G, B = case["grid"], case.get("batch", 1)
    c = (np.arange(G) + 0.5) / G - 0.5
    r = np.sqrt(c[:, None, None] ** 2 + c[None, :, None] ** 2 + c[None, None, :] ** 2)
    div, mask, sol, scale = [], [], [], []
    for _ in range(B):
        level = case.get("level", 0.3) * rng.uniform(0.9, 1.1)
        m = (np.abs(r - level) < 3.0 / G).astype(np.float32)
        s = float(rng.uniform(50, 200))
        d = (m * (r - level) * G + 0.3 * m * rng.standard_normal((G, G, G))).astype(np.float32)
        d *= np.float32(s / math.sqrt(float((d ** 2).sum()) / m.sum()))
        div.append(d)
        mask.append(m)
        sol.append((m * s * (level - r) * G * 0.5 + m * s * 0.1 * rng.standard_normal((G, G, G))).astype(np.float32))
        scale.append(s)
    return np.stack(div), np.stack(mask), np.stack(sol), np.array(scale, np.float32)


def _mesh_buffers(shape, depth, pinned):
    """Zeroed host buffers with room for more than such a surface has."""
    cells = AREA[shape] * 4 ** depth
    v = torch.zeros(int(5 * cells) + 100000, 3, dtype=torch.float32, pin_memory=pinned)
    t = torch.zeros(int(8 * cells) + 200000, 3, dtype=torch.int32, pin_memory=pinned)
    return v, t


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("mesh", "field"):
        p, n = _cloud(case["shape"], case["points"], seed)
        s = {"kind": kind, "n": len(p), "g": prg.Reconstructor(max_depth=case["depth"])}
        source = case.get("source", "host")
        if source == "device":
            s["p"], s["nrm"] = torch.from_numpy(p).cuda(), torch.from_numpy(n).cuda()
            torch.cuda.synchronize()
        elif source == "pinned":
            s["keep"] = _pinned(p), _pinned(n)
            s["p"], s["nrm"] = (t.numpy() for t in s["keep"])
        else:
            s["p"], s["nrm"] = p, n
        s["device"] = source == "device"
        if kind == "mesh":
            s["subdivide"] = case["subdivide"]
            s["v"], s["t"] = _mesh_buffers(case["shape"], case["depth"], case["sink"] == "pinned")
        else:
            rows = sum(min(8 * len(p), 8 ** d) for d in range(case["depth"] + 1))  # at most
            s["keys"], s["solution"] = np.zeros(rows, np.uint32), np.zeros(rows, np.float32)
            s["values"] = np.zeros(len(p), np.float32)
        return s
    if kind == "batch":
        sizes = _batch_sizes(case)
        depths = [_usual_depth(n) for n in sizes]
        return {"kind": kind, "clouds": [_cloud("superquadrics", n, 100 * seed + i) for i, n in enumerate(sizes)],
                "depths": depths, "meshes": [_mesh_buffers("superquadrics", d, False) for d in depths]}
    if kind == "weld":
        v, t, n_leaf = _planted_mesh(case, seed)
        return {"kind": kind, "g": prg.Reconstructor(max_depth=5),
                "mesh": prg.Mesh(v, t, np.zeros(3, np.float32), 1.0, n_leaf, len(t))}
    net = prg.UNet(grid=case["grid"], seed=1)
    net.set_params(_net_params(seed))
    return {"kind": kind, "net": net, "data": _samples(case, seed)}


# ---- one pass -------------------------------------------------------------------------
def _points_to_solution(s):
    g = s["g"]
    if s["device"]:
        g._call("prg_set_points", C.c_void_p(s["p"].data_ptr()), C.c_void_p(s["nrm"].data_ptr()), s["n"], 1)
    else:
        g.set_points(s["p"], s["nrm"])
    g.build_octree()
    g.compute_divergence()
    return g.solve()


def run(s):
    kind = s["kind"]
    if kind == "mesh":
        g = s["g"]
        stats = _points_to_solution(s)
        g._call("prg_isovalue", None)  # stays on the device for the mesh
        m = prg.PrgMesh()
        g._call("prg_extract_mesh_into", int(s["subdivide"]), C.c_void_p(s["v"].data_ptr()), s["v"].numel(),
                C.c_void_p(s["t"].data_ptr()), s["t"].numel(), C.byref(m))
        # the buffers whole (zeros past the mesh), and what they hold
        return {"vertices": s["v"], "triangles": s["t"], "center": np.array(m.center[:], np.float32),
                "scale": float(m.scale), "iters": np.array([x["iters"] for x in stats], np.int64),
                "counts": np.array([m.n_vertices, m.n_triangles, m.n_leaf_vertices, m.n_leaf_triangles], np.int64)}
    if kind == "field":
        g = s["g"]
        _points_to_solution(s)
        iso = g.isovalue()
        center, scale = g.transform()
        counts, _ = g.level_info()
        nbytes = 4 * int(counts.sum())
        for which, buf, size in ((prg.BUF_KEY, s["keys"], nbytes), (prg.BUF_SOLUTION, s["solution"], nbytes),
                                 (prg.BUF_POINT_VALUES, s["values"], s["values"].nbytes)):
            g._call("prg_read_buffer", which, C.c_void_p(buf.ctypes.data), size)
        return {"center": center, "scale": scale, "counts": counts, "iso": iso, "keys": s["keys"],
                "solution": s["solution"], "values": s["values"]}
    if kind == "batch":
        st, res = prg.reconstruct_batch(s["clouds"], s["depths"], concurrency=4, return_meshes=True)
        for (v, t), r in zip(s["meshes"], res):  # collected in the program's own buffers
            v[: r["vertices"]] = torch.from_numpy(r["mesh_vertices"])
            t[: r["triangles"]] = torch.from_numpy(r["mesh_triangles"])
        return {"status": st, "counts": np.array([[r[k] for k in ("status", "vertices", "triangles", "total_iters")]
                                                  for r in res], np.int64), "meshes": s["meshes"]}
    if kind == "weld":
        m, removed = s["g"].weld_mesh(s["mesh"])
        return {"vertices": m.vertices, "triangles": m.triangles, "leaf": m.n_leaf_vertices, "removed": removed}
    div, mask, sol, scale = s["data"]
    if kind == "predict":
        return s["net"].predict(div[0], mask[0], float(scale[0]))
    loss = s["net"].train_step(div, mask, sol, scale, 1e-3)
    return {"loss": loss, "params": s["net"].get_params()}


# ---- what a pass cannot do without ------------------------------------------------------
def _cloud_work(shape, n, depth, subdivide):
    cells = AREA[shape] * 4 ** depth  # depth-D cells of the surface, up to its slope
    if not subdivide:
        cells = min(cells, 2 * n)
    rows = sum(min(5.3 * AREA[shape] * 4 ** d, 8 * n, 8 ** d) for d in range(depth + 1))
    # points and normals in, about 1.6 vertices and 3 triangles per cell out;
    # about 20 conjugate-gradient iterations of a 27-point stencil per depth
    return {"bytes": 24 * n + 12 * 4.6 * cells, "flops": 20 * 54 * rows}


def work(case):
    kind = case["kind"]
    if kind == "mesh":
        return _cloud_work(case["shape"], case["points"], case["depth"], case["subdivide"])
    if kind == "field":
        w = _cloud_work(case["shape"], case["points"], case["depth"], False)
        rows = w["flops"] / (20 * 54)
        return {"bytes": 28 * case["points"] + 8 * rows, "flops": w["flops"]}
    if kind == "batch":
        parts = [_cloud_work("superquadrics", n, _usual_depth(n), True) for n in _batch_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "weld":
        return {"bytes": 2 * 12 * (case["vertices"] + case["triangles"]), "flops": 0}
    G = case["grid"]
    flops = sum(54 * i * o * (G >> lv) ** 3 for (i, o), lv in zip(CONVS, LEVEL)) + 32 * G ** 3
    if kind == "predict":
        return {"bytes": 12 * G ** 3 + 4 * _num_params(), "flops": flops}
    return {"bytes": case["batch"] * 12 * G ** 3 + 16 * _num_params(), "flops": 3 * flops * case["batch"]}


# ---- the same outputs in 64 bits ---------------------------------------------------------
def _conv(a, w, b):
    """3x3x3 convolution (zero padding) and ReLU; a: (G, G, G, Cin), w: (27, Cout, Cin)."""
    G, _, _, ci = a.shape
    p = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b
    for t in range(27):
        x, y, z = t // 9, (t // 3) % 3, t % 3
        out = out + p[x:x + G, y:y + G, z:z + G].reshape(-1, ci) @ w[t].T.contiguous()
    return torch.relu(out).reshape(G, G, G, -1)


def _pool(a):
    G = a.shape[0] // 2
    return a.reshape(G, 2, G, 2, G, 2, -1).mean(dim=(1, 3, 5))


def _up(a):
    G, c = a.shape[0], a.shape[3]
    return a[:, None, :, None, :, None].expand(G, 2, G, 2, G, 2, c).reshape(2 * G, 2 * G, 2 * G, c)


def _net(params, div, mask, scale):
    """The network's prediction in units of `scale`; params: the flat vector, float64."""
    o, conv = 0, []
    for i, c in CONVS:
        w = params[o:o + 27 * i * c].reshape(27, c, i)
        o += 27 * i * c
        conv.append((w, params[o:o + c]))
        o += c
    x = torch.zeros(*div.shape, 16, dtype=torch.float64, device=div.device)
    x[..., 0] = div / scale
    x[..., 1] = mask
    e0 = _conv(_conv(x, *conv[0]), *conv[1])
    e1 = _conv(_conv(_pool(e0), *conv[2]), *conv[3])
    e2 = _conv(_conv(_pool(e1), *conv[4]), *conv[5])
    b = _conv(_conv(_pool(e2), *conv[6]), *conv[7])
    d2 = _conv(_conv(torch.cat([_up(b), e2], 3), *conv[8]), *conv[9])
    d1 = _conv(_conv(torch.cat([_up(d2), e1], 3), *conv[10]), *conv[11])
    d0 = _conv(_conv(torch.cat([_up(d1), e0], 3), *conv[12]), *conv[13])
    return d0 @ params[o:o + 16] + params[o + 16]


def _weld(v, t, n_leaf):
    _, first, inverse = np.unique(v.view(np.uint32), axis=0, return_index=True, return_inverse=True)
    owner = first[inverse.reshape(-1)]  # the first vertex with the same bits
    keep = owner == np.arange(len(v))
    number = np.cumsum(keep) - 1
    return {"vertices": v[keep].astype(np.float64), "triangles": number[owner[t]], "leaf": int(keep[:n_leaf].sum()),
            "removed": int((~keep).sum())}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mesh", "field"):
        # the normalisation; the octree's functions and the solve need the
        # whole method, which plain numpy does not give in seconds
        if case.get("shape") != "sphere" or case["points"] > 100000:
            return None
        p, _ = _cloud(case["shape"], case["points"], seed)
        lo, hi = p.min(0).astype(np.float64), p.max(0).astype(np.float64)
        return {"center": None, "scale": float(1.25 * (hi - lo).max())}
    if kind == "weld":
        return _weld(*_planted_mesh(case, seed))
    if kind not in ("predict", "train"):
        return None
    div, mask, sol, scale = (torch.from_numpy(a.astype(np.float64)).cuda() for a in _samples(case, seed))
    params = torch.from_numpy(_net_params(seed).astype(np.float64)).cuda()
    if kind == "predict":
        with torch.no_grad():
            return _net(params, div[0], mask[0], scale[0]) * scale[0]
    params.requires_grad_(True)
    total = 0.0
    B = len(scale)
    for k in range(B):
        d = _net(params, div[k], mask[k], scale[k]) - sol[k] / scale[k]
        loss = (mask[k] * d * d).sum() / mask[k].sum() / B
        loss.backward()
        total += float(loss.detach())
    # the first Adam step: both moments hold this gradient alone
    g = params.grad
    return {"loss": total, "params": params.detach() - 1e-3 * g / (g.abs() + 1e-8)}
