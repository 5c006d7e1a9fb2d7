"""The learned warm start's U-Net on the GPU (BF16 matrix-core convolutions,
FP32 accumulation) against its numpy oracle (oracle/unet_ref.py, which
mirrors the GPU's BF16 rounding points and accumulates in float64), and
the warm start inside the solver."""
import numpy as np
import pytest

from oracle import unet_ref as U

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


def _sample(G, seed):
    rng = np.random.default_rng(seed)
    b = rng.standard_normal((G, G, G)).astype(np.float32)
    m = (rng.random((G, G, G)) < 0.4).astype(np.float32)
    t = rng.standard_normal((G, G, G)).astype(np.float32)
    return b, m, t


@pytest.fixture(scope="module")
def net16(prg):
    net = prg.UNet(grid=16, seed=7)
    p = net.get_params()
    assert p.size == U.num_params()
    d = U.unflatten(p)
    rng = np.random.default_rng(3)
    for k in d:
        if k.endswith(".b"):
            d[k] = (rng.standard_normal(d[k].shape) * 0.05).astype(np.float32)
    net.set_params(U.flatten(d))
    yield net, d
    net.close()


def test_forward_matches_oracle(net16):
    net, d = net16
    print("\n[unet forward G=16]", flush=True)
    b, m, _ = _sample(16, 1)
    x = np.zeros((16, 16, 16, U.CIN0), np.float32)
    x[..., 0] = b
    x[..., 1] = m
    ref, _ = U.forward(d, x)
    out = net.predict(b, m, 1.0)
    err = _rel(out, ref)
    print(f"prediction rel L2 {err:.2e}")
    assert err <= 2e-3


def test_gradients_match_oracle(net16):
    net, d = net16
    print("\n[unet gradients G=16]", flush=True)
    b, m, t = _sample(16, 2)
    x = np.zeros((16, 16, 16, U.CIN0), np.float32)
    x[..., 0] = b
    x[..., 1] = m
    loss_ref, grads_ref, _ = U.loss_and_grad(d, x, t, m)
    loss, g = net.gradients(b, m, t, 1.0)
    assert abs(loss - loss_ref) <= 1e-3 * abs(loss_ref)
    gd = U.unflatten(g)
    worst = 0.0
    for name, _ in U.param_layout():
        err = _rel(gd[name], grads_ref[name])
        worst = max(worst, err)
        assert err <= 3e-2, (name, err)
    print(f"loss {loss:.6f} (oracle {loss_ref:.6f}); worst gradient rel L2 {worst:.2e}")


def test_training_reduces_loss(prg):
    print("\n[unet training G=16]", flush=True)
    net = prg.UNet(grid=16, seed=11)
    try:
        rng = np.random.default_rng(5)
        G = 16
        B = 4
        # a learnable map: the target is a smoothed copy of the input on the mask
        bs = rng.standard_normal((B, G, G, G)).astype(np.float32)
        ms = np.ones((B, G, G, G), np.float32)
        ts = 0.5 * (bs + np.roll(bs, 1, axis=1) + np.roll(bs, -1, axis=2)) / 3.0
        first = net.train_step(bs, ms, ts, np.ones(B, np.float32), 2e-3)
        for _ in range(80):
            last = net.train_step(bs, ms, ts, np.ones(B, np.float32), 2e-3)
        print(f"loss {first:.4f} -> {last:.4f}")
        assert last < 0.6 * first
    finally:
        net.close()


def test_learned_warm_start_solves_to_tolerance(prg):
    print("\n[warm start: sphere N=35947 D=7, network on depth 5]", flush=True)
    p, n = prg.synth_sphere(35947, 1)
    net = prg.UNet(grid=32, seed=3)
    plain = prg.Reconstructor(max_depth=7)
    warm = prg.Reconstructor(max_depth=7, warm_start=prg.WARM_LEARNED)
    try:
        warm.set_warm_start_net(net)
        for g in (plain, warm):
            g.set_points(p, n)
            g.build_octree()
            g.compute_divergence()
        sp, sw = plain.solve(), warm.solve()
        for s in sp + sw:
            assert s["true_rel_residual"] <= 2e-6
        # the untrained network's start changes the depth-5 trajectory only
        assert [s["iters"] for s in sp][:5] == [s["iters"] for s in sw][:5]
        assert [s["iters"] for s in sp][6:] == [s["iters"] for s in sw][6:]
        xw = warm.read_buffer(prg.BUF_SOLUTION)
        xp = plain.read_buffer(prg.BUF_SOLUTION)
        counts, bases = plain.level_info()
        sl = slice(int(bases[5]), int(bases[5] + counts[5]))
        assert _rel(xw[sl], xp[sl]) <= 1e-4
    finally:
        warm.close()
        plain.close()
        net.close()


@pytest.mark.parametrize("grid", [16, 64])
def test_worse_than_zero_warm_start_falls_back(prg, monkeypatch, grid):
    """A warm start with ||b - A x0|| > ||b|| is replaced by x0 = 0: with the
    prediction scaled by 1e6 (test setting PRG_WARM_START_SCALE), the solve
    equals the plain solve bit for bit, and prg_warm_start_info reports the
    rejection.  grid 16 warm-starts depth 4 (the one-workgroup small-depth
    CG), grid 64 depth 6 (the multi-kernel CG of the large depths)."""
    print(f"\n[warm start fallback: sphere N=35947 D=8, network grid {grid}]", flush=True)
    p, n = prg.synth_sphere(35947, 1)
    net = prg.UNet(grid=grid, seed=3)
    plain = prg.Reconstructor(max_depth=8)
    monkeypatch.setenv("PRG_WARM_START_SCALE", "1e6")
    warm = prg.Reconstructor(max_depth=8, warm_start=prg.WARM_LEARNED)
    try:
        warm.set_warm_start_net(net)
        for g in (plain, warm):
            g.set_points(p, n)
            g.build_octree()
            g.compute_divergence()
        counts, _ = plain.level_info()
        wd = {16: 4, 64: 6}[grid]
        assert (counts[wd] > 2048) == (grid == 64), counts.tolist()
        sp, sw = plain.solve(), warm.solve()
        assert warm.warm_start_info() == (wd, True)
        assert [s["iters"] for s in sp] == [s["iters"] for s in sw]
        assert np.array_equal(plain.read_buffer(prg.BUF_SOLUTION).view(np.uint32),
                              warm.read_buffer(prg.BUF_SOLUTION).view(np.uint32))
        assert plain.warm_start_info() == (-1, False)
    finally:
        warm.close()
        plain.close()
        net.close()


def _torch_gradients(params, b, m, t):
    """oracle.unet_ref's loss and gradient (the same BF16 rounding points) in
    float32 torch on the CPU, fast enough for 128^3; one 2-D product per tap."""
    import torch
    import torch.nn.functional as F

    def bf16(a):
        return a.bfloat16().float()

    def taps(p, G):
        for k in range(27):
            x, y, z = k // 9, (k // 3) % 3, k % 3
            yield k, p[x:x + G, y:y + G, z:z + G]

    class Conv(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a, w):
            G, ci = a.shape[0], a.shape[3]
            p, wb = F.pad(bf16(a), (0, 0, 1, 1, 1, 1, 1, 1)), bf16(w)
            ctx.save_for_backward(p, wb)
            return sum(s.reshape(-1, ci) @ wb[k].T for k, s in taps(p, G)).reshape(G, G, G, -1)

        @staticmethod
        def backward(ctx, g):
            p, wb = ctx.saved_tensors
            G, ci, co = g.shape[0], p.shape[3], g.shape[3]
            gb = bf16(g)
            dw = torch.stack([gb.reshape(-1, co).T @ s.reshape(-1, ci) for _, s in taps(p, G)])
            gp = F.pad(gb, (0, 0, 1, 1, 1, 1, 1, 1))
            da = sum(s.reshape(-1, co) @ wb[26 - k] for k, s in taps(gp, G)).reshape(G, G, G, ci)
            return da, dw

    flat = torch.from_numpy(params).requires_grad_(True)
    conv, o = [], 0
    for _, ci, co in U.CONVS:
        conv.append((flat[o:o + 27 * ci * co].reshape(27, co, ci), flat[o + 27 * ci * co:o + 27 * ci * co + co]))
        o += 27 * ci * co + co

    def run(k, a):
        return torch.relu(Conv.apply(a, conv[k][0]) + conv[k][1])

    def pool(a):
        H = a.shape[0] // 2
        return a.reshape(H, 2, H, 2, H, 2, -1).mean(dim=(1, 3, 5))

    def up(a):
        H, c = a.shape[0], a.shape[3]
        return a[:, None, :, None, :, None].expand(H, 2, H, 2, H, 2, c).reshape(2 * H, 2 * H, 2 * H, c)

    db, dm, dt = (torch.from_numpy(a) for a in (b, m, t))
    x = torch.stack([db, dm] + [torch.zeros_like(db)] * 14, dim=3)
    e0 = run(1, run(0, x))
    e1 = run(3, run(2, pool(e0)))
    e2 = run(5, run(4, pool(e1)))
    bt = run(7, run(6, pool(e2)))
    d2 = run(9, run(8, torch.cat([up(bt), e2], 3)))
    d1 = run(11, run(10, torch.cat([up(d2), e1], 3)))
    d0 = run(13, run(12, torch.cat([up(d1), e0], 3)))
    pred = d0 @ flat[o:o + 16] + flat[o + 16]
    loss = (dm * (pred - dt) ** 2).sum() / dm.sum()
    loss.backward()
    return float(loss.detach()), flat.grad.numpy()


@pytest.mark.parametrize("grid", [32, 64, 128])
def test_gradients_on_larger_grids(prg, grid):
    """Every level's weight-gradient instance (grids 4 to 128; 16 and 2 are in
    the 16^3 test above), with that test's tolerance: the rounding points are
    the same, so only BF16 roundings and ReLU masks that flip by an
    accumulation's last bits differ.  A lost tap, row or halo is over 0.1."""
    print(f"\n[unet gradients G={grid}]", flush=True)
    b, m, t = _sample(grid, 20 + grid)
    net = prg.UNet(grid=grid, seed=7)
    try:
        loss_ref, ref = _torch_gradients(net.get_params(), b, m, t)
        loss, g = net.gradients(b, m, t, 1.0)
    finally:
        net.close()
    assert abs(loss - loss_ref) <= 1e-3 * abs(loss_ref)
    gd, rd = U.unflatten(g), U.unflatten(ref)
    for name, _ in U.param_layout():
        err = _rel(gd[name], rd[name])
        assert err <= 3e-2, (name, err)


@pytest.mark.parametrize("batch", [1, 3, 18])
def test_train_step_is_one_adam_step_on_the_mean_gradient(prg, batch):
    """Samples that share launches (18: two launches of 16 and 2) give the sum
    of their single gradients.  The first Adam step is lr g / (|g| + eps):
    with float moments, divisions and a parameter below 2 the result is
    within 1e-6 lr + 2^-23 of it where |g| is far above eps."""
    print(f"\n[unet train step G=16 batch {batch}]", flush=True)
    lr, G = 1e-3, 16
    net = prg.UNet(grid=G, seed=13)
    try:
        s = [_sample(G, 40 + k) for k in range(batch)]
        scales = np.linspace(0.5, 2.0, batch).astype(np.float32)
        p0 = net.get_params()
        losses, grads = zip(*[net.gradients(b, m, t, float(f)) for (b, m, t), f in zip(s, scales)])
        g = np.sum(np.array(grads, np.float64), axis=0) / batch
        loss = net.train_step(*(np.stack(a) for a in zip(*s)), scales, lr)
        p1 = net.get_params()
    finally:
        net.close()
    assert abs(loss - np.mean(losses)) <= 1e-12 * abs(np.mean(losses))
    big = np.abs(g) > 1e-3 * np.abs(g).max()  # (sums of up to 18 floats: signs are certain here)
    assert big.any()
    want = p0 - lr * np.sign(g)
    assert np.abs(p1 - want)[big].max() <= 1e-6 * lr + 2.0 ** -23 + lr * 1e-8 / np.abs(g[big]).min()
    assert np.abs(p1 - p0).max() <= lr * (1 + 1e-5) + 2.0 ** -23
