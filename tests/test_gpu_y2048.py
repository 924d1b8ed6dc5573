"""The inverse y transform of length 2048 at the sizes where its tile changes:
8-column split tiles from 256 workgroups on, 4-column tiles below; whole tiles
and a last tile of one column."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


# (n0, n1, n2), periodic y: workgroups of 8 columns = ceil((n2 + 1) / 8) n0 3
@pytest.mark.parametrize("n,pbc", [((44, 1024, 8), (0, 0, 0)),   # 264, last tile one column
                                   ((43, 1024, 7), (0, 0, 0)),   # 129: below
                                   ((86, 1024, 7), (0, 0, 0)),   # 258, whole tiles only
                                   ((44, 2048, 8), (0, 1, 0))])  # 264, every row holds data
def test_field(n, pbc):
    import mmx
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    cell = (3e-9, 3e-9, 4e-9)
    print("[case]", n, pbc, flush=True)
    plan = mmx.DemagPlan(n, cell, pbc)
    kh, _ = O.kernel_fft(plan.p, K9=O.kernel_arne(plan.p, cell, pbc))
    m = O.normalize(np.random.default_rng(sum(n)).normal(size=(3,) + n)).astype(np.float32)
    want = O.MU0 * 8e5 * O.demag_conv(n, plan.p, kh, m.astype(np.float64))
    dm = torch.from_numpy(m).cuda()
    db = torch.empty_like(dm)
    plan.update_b(db.data_ptr(), dm.data_ptr(), 8e5)
    torch.cuda.synchronize()
    # the repository's parity bar for fields, relative to the largest value
    assert np.abs(db.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()
