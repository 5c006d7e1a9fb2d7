"""Training steps of several samples against Adam on the gradients of single
samples (prg_unet_gradients).  Two steps of different batch sizes: the second
one's m / sqrt(v) depends on the ratio of the two mean gradients, so a wrong
weight of a batch or of one of its samples shows, which a first step (lr times
the gradient's sign) hides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # float32 rounding


def _samples(grid, n, seed):
    rng = np.random.default_rng(seed)
    b, m, t = (rng.standard_normal((n, grid, grid, grid)).astype(np.float32) for _ in range(3))
    return b, (m > 0.3).astype(np.float32), t, np.linspace(0.5, 2.0, n).astype(np.float32)


def _mean_gradient(net, s):
    """The mean of the single gradients, and a bound on the error of the
    library's: a float sum of n terms and a multiplication by 1 / n."""
    g = np.array([net.gradients(b, m, t, float(f))[1] for b, m, t, f in zip(*s)], np.float64)
    return g.mean(axis=0), (len(g) + 2) * U * np.abs(g).mean(axis=0)


@pytest.mark.parametrize("grid,first,second", [(16, 18, 2), (32, 3, 5), (64, 8, 2)])
def test_two_training_steps_are_adam_on_single_gradients(prg, grid, first, second):
    print(f"\n[unet training, G={grid}, batches of {first} and {second}]", flush=True)
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 1e-8
    s1, s2 = _samples(grid, first, grid), _samples(grid, second, grid + 1)
    net = prg.UNet(grid=grid, seed=17)
    try:
        g1, e1 = _mean_gradient(net, s1)
        net.train_step(*s1, lr)
        g2, e2 = _mean_gradient(net, s2)
        p1 = net.get_params().astype(np.float64)
        net.train_step(*s2, lr)
        p2 = net.get_params().astype(np.float64)
    finally:
        net.close()
    a1, a2 = b1 * (1 - b1), 1 - b1
    w1, w2 = b2 * (1 - b2), 1 - b2
    m, v = a1 * g1 + a2 * g2, w1 * g1 ** 2 + w2 * g2 ** 2
    c1, c2 = 1 - b1 ** 2, 1 - b2 ** 2
    s = np.sqrt(v / c2)
    want = p1 - lr * (m / c1) / (s + eps)
    # where float squares neither underflow nor leave their rounding behind
    ok = v > 1e-22
    # parameters that no sample of either step reaches stay where they are
    still = (e1 == 0) & (e2 == 0)
    assert np.array_equal(p2[still], p1[still])
    with np.errstate(divide="ignore", invalid="ignore"):
        # gradients off by e1, e2; constants rounded to float, and five roundings
        # of each moment's terms
        dm = a1 * e1 + a2 * e2 + 6 * U * (a1 * np.abs(g1) + a2 * np.abs(g2))
        dv = 2 * (w1 * np.abs(g1) * e1 + w2 * np.abs(g2) * e2) + 8 * U * v
        # through m / sqrt(v): relative errors add, half of v's; eight roundings
        # of the step, one of the result
        rel = 0.5 * dv / v
        bound = lr / c1 * (dm / s + np.abs(m) / s * (1.1 * rel + 8 * U)) + U * np.abs(want)
    ok &= rel < 0.05
    err = np.abs(p2 - want)
    print(f"  parameters {ok.sum()} of {ok.size}, largest error {err[ok].max():.2e} of steps up to "
          f"{np.abs(want - p1)[ok].max():.2e}, largest share of its bound {(err[ok] / bound[ok]).max():.2f}", flush=True)
    assert (ok | still).mean() > 0.9
    assert (err[ok] <= bound[ok]).all()
