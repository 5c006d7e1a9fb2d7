"""A training call that failed leaves nothing queued that reaches into the next
one: the next call's loss and weights are those of a network that saw no
failure, also from pinned arrays, whose copies a call does not wait for."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pinned(prg, a):
    """A copy of a in pinned memory (kept until the process ends)."""
    p = C.c_void_p()
    hip = prg.lib()  # (the runtime is among the library's dependencies)
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    assert hip.hipHostMalloc(C.byref(p), a.nbytes, 0) == 0
    out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), shape=(a.size,)).reshape(a.shape)
    out[...] = a
    return out


def _batch(prg, grid, batch, seed):
    rng = np.random.default_rng(seed)
    b, m, t = (rng.standard_normal((batch, grid, grid, grid)).astype(np.float32) for _ in range(3))
    m = (m > 0.0).astype(np.float32)
    return [_pinned(prg, a) for a in (b, m, t)], np.full(batch, 0.25, np.float32)


@pytest.mark.parametrize("grid,batch", [(16, 3), (64, 8)])
def test_call_after_a_failed_one(prg, monkeypatch, grid, batch):
    first, scales = _batch(prg, grid, batch, 1)
    second, _ = _batch(prg, grid, batch, 2)
    plain = prg.UNet(grid=grid, seed=3)
    loss = plain.train_step(*second, scales, 1e-3)
    want = plain.get_params()
    monkeypatch.setenv("PRG_UNET_FAIL_CALL", "1")
    net = prg.UNet(grid=grid, seed=3)
    monkeypatch.delenv("PRG_UNET_FAIL_CALL")
    print(f"\n[a failed training call, then one that must not see it: G={grid} batch {batch}]", flush=True)
    with pytest.raises(prg.PrgError) as e:
        net.train_step(*first, scales, 1e-3)
    assert e.value.status == prg.E_HIP
    assert net.train_step(*second, scales, 1e-3) == loss
    assert np.array_equal(net.get_params().view(np.uint32), want.view(np.uint32))
    net.close()
    plain.close()
