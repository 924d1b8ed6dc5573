"""The surrogate's backward pass where its split changes, and its update.

The weight gradients take one workgroup per 16 x 16 pixel tile up to 128
tiles and several tiles per workgroup beyond; the reduction of the partial
gradients also makes the Adam step and the new bf16 weights.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import surrogate as OS  # noqa: E402

CELL = (3e-9, 4e-9, 4e-9)


def _sur(n):
    import torch
    import mmx
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    mmx.check(mmx.lib().mmx_init(0))
    sim = mmx.Sim(n, CELL)
    sim.setv("Msat", 8e5)
    sim.setv("Aex", 1.3e-11)
    sim.setv("alpha", 0.02)
    return mmx, sim, mmx.Surrogate(sim, seed=1)


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


# 8 x 16 tiles: the last grid with a tile each; 11 x 12: two for some workgroups
@pytest.mark.parametrize("n", [(1, 128, 256), (1, 176, 192)])
def test_gradients_by_tiles(n):
    """Same bounds as the small grids' comparison: the sums are FP32 over
    products of bf16 values rounded at the oracle's points.  A tile left out
    or taken twice changes a gradient of independent pixels by 9 %."""
    mmx, sim, sur = _sur(n)
    rng = np.random.default_rng(n[1])
    Ws, bs = OS.init_params(seed=5, n0=1)
    Ws[3] *= 10.0
    sur.set_params(mmx.Surrogate.flatten(Ws, bs))
    Ws, bs = mmx.Surrogate.unflatten(sur.get_params())
    x = np.zeros((n[1], n[2], 32))
    x[:, :, :8] = rng.normal(size=(n[1], n[2], 8))
    tgt = rng.normal(size=(n[1], n[2], 3)) * 0.3
    out_g, loss_g = sur.net(x, tgt)
    out_o, acts = OS.forward(Ws, bs, OS.bf16(x))
    loss_o, gout = OS.loss_and_grad_out(out_o, tgt, 3)
    dWs, dbs = OS.backward(Ws, acts, gout)
    assert _rel(out_g, out_o) < 5e-3
    assert abs(loss_g - loss_o) < 1e-2 * loss_o
    gW, gb = mmx.Surrogate.unflatten(sur.get_grads())
    for l in range(4):
        used = slice(None) if l else slice(0, 8)
        assert _rel(gW[l][:, :, used], dWs[l][:, :, used]) < 2e-2
        assert _rel(gb[l][:3] if l == 3 else gb[l], dbs[l][:3] if l == 3 else dbs[l]) < 2e-2


def test_update_and_new_weights():
    """One train step from zero moments moves a parameter with gradient g by
    lr g / (|g| + eps); the next forward pass uses the new weights."""
    import torch
    n = (2, 32, 48)
    mmx, sim, sur = _sur(n)
    rng = np.random.default_rng(8)
    m = rng.normal(size=(3,) + n)
    m = torch.from_numpy((m / np.linalg.norm(m, axis=0)).astype(np.float32)).cuda()
    w0 = sur.get_params().astype(np.float64)
    lr = 1e-2
    sur.train_step(m.data_ptr(), lr=lr)
    w1, g = sur.get_params(), sur.get_grads().astype(np.float64)
    # FP32 rounding of a handful of operations, of the step and of the sum
    assert np.abs(w1 - (w0 - lr * g / (np.abs(g) + 1e-8))).max() < 1e-5 * lr + 2e-7 * np.abs(w0).max()
    x = np.zeros((n[1], n[2], 32))
    x[:, :, :14] = rng.normal(size=(n[1], n[2], 14))
    out = sur.net(x)
    out = out[0] if isinstance(out, tuple) else out
    Ws, bs = mmx.Surrogate.unflatten(w1)
    assert _rel(out, OS.forward(Ws, bs, OS.bf16(x))[0]) < 5e-3
