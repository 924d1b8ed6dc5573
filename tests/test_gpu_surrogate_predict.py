"""A prediction is the network on the packed (m, coarse B, position) channels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402

MU0MS = O.MU0 * 8e5


@pytest.mark.parametrize("n", [(1, 16, 16), (2, 32, 48), (5, 48, 16)])
def test_prediction_is_the_net_on_its_channels(n):
    import torch
    import mmx
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    mmx.check(mmx.lib().mmx_init(0))
    print("predict", n, flush=True)
    sim = mmx.Sim(n, (3e-9, 4e-9, 4e-9))
    for k, v in (("Msat", 8e5), ("Aex", 1.3e-11), ("alpha", 0.02)):
        sim.setv(k, v)
    sur = mmx.Surrogate(sim, seed=4)
    m = O.normalize(np.random.default_rng(n[1]).normal(size=(3,) + n)).astype(np.float32)
    dm = torch.from_numpy(m).cuda()
    coarse, full = torch.empty_like(dm), torch.empty_like(dm)
    sur.predict_b(dm.data_ptr(), coarse.data_ptr(), coarse_only=True)
    sur.predict_b(dm.data_ptr(), full.data_ptr())
    torch.cuda.synchronize()
    coarse, full = coarse.cpu().numpy(), full.cpu().numpy()
    n0, P = n[0], n[1:]
    x = np.zeros(P + (32,), np.float32)
    x[..., :3 * n0] = m.reshape((3 * n0,) + P).transpose(1, 2, 0)
    x[..., 3 * n0:6 * n0] = coarse.reshape((3 * n0,) + P).transpose(1, 2, 0) / MU0MS
    x[..., 6 * n0] = np.where(np.arange(P[0]) & 1, 1.0, -1.0)[:, None]
    x[..., 6 * n0 + 1] = np.where(np.arange(P[1]) & 1, 1.0, -1.0)[None, :]
    out = sur.net(x)[..., :3 * n0].transpose(2, 0, 1).reshape((3,) + n)
    got = (full.astype(np.float64) - coarse) / MU0MS
    # the bar of the net's comparison with its oracle: the coarse B's last place
    # can flip a bf16 rounding
    assert np.linalg.norm(got - out) < 5e-3 * np.linalg.norm(out)
