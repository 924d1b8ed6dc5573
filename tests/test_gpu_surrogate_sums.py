"""Sums of the surrogate's training step over inputs whose sum is exact: terms
that a float32 accumulator loses once it holds a large one, and that the sums by
tile (bias gradients) and in 64 bits (the loss) keep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _zero_net(n):
    import torch
    import mmx
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    mmx.check(mmx.lib().mmx_init(0))
    sim = mmx.Sim(n, (3e-9, 4e-9, 4e-9))
    for k, v in (("Msat", 8e5), ("Aex", 1.3e-11), ("alpha", 0.02)):
        sim.setv(k, v)
    sur = mmx.Surrogate(sim, seed=1)
    sur.set_params(np.zeros(sur.nparams, np.float32))   # out = 0, so d = -target
    return mmx, sim, sur


# pixels that one partial sum of the loss covers: two of a wave, and two of one
# thread where the grid has more pixels than the launch has threads
@pytest.mark.parametrize("n,other", [((1, 32, 64), 32), ((1, 512, 512), 65536)])
def test_loss_keeps_small_terms(n, other):
    mmx, sim, sur = _zero_net(n)
    tgt = np.zeros((n[1] * n[2], 3), np.float32)
    tgt[0, 0], tgt[other, 0] = 1.0, 2.0 ** -13
    _, loss = sur.net(np.zeros((n[1], n[2], 32), np.float32), tgt.reshape(n[1], n[2], 3))
    # (1 + 2^-26) over sum target^2, which rounds to 1 in float32
    assert loss == 1.0 + 2.0 ** -26


# tiles of 16 x 16 pixels; 128 workgroups, so tile 128 follows tile 0
def test_bias_gradient_keeps_small_tiles():
    n = (1, 256, 256)
    mmx, sim, sur = _zero_net(n)
    tgt = np.zeros((n[1], n[2], 3), np.float32)
    tgt[0:16, 0:16, 0] = -1.0               # tile 0
    tgt[128:144, 0:16, 0] = -2.0 ** -19     # tile 128
    sur.net(np.zeros((n[1], n[2], 32), np.float32), tgt)
    _, gb = mmx.Surrogate.unflatten(sur.get_grads())
    # gradient scale 2 / 256; every sum by tile is representable
    assert gb[3][0] == 2.0 + 2.0 ** -18
