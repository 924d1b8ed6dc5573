"""Construction of the demag kernel: the near-field table of Kernel_Arne and the
FP64 transform's line tiles at the sizes where they change shape."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mmx():
    import mmx
    mmx.check(mmx.lib().mmx_init(0))
    return mmx


# near table: smaller and larger than the grid, cells of aspect 4, one point per
# axis everywhere, periodic images inside and outside of it
NEAR = [((2, 24, 30), (3e-9, 3e-9, 3e-9), (0, 0, 0), 6),
        ((1, 12, 40), (1e-9, 4e-9, 2e-9), (0, 0, 0), 6),
        ((3, 20, 6), (4e-9, 1e-9, 4e-9), (0, 0, 0), 3),
        ((2, 10, 12), (3e-9, 3e-9, 3e-9), (0, 0, 0), 1),
        ((2, 6, 24), (3e-9, 3e-9, 3e-9), (0, 1, 1), 6),
        ((4, 8, 6), (2e-9, 4e-9, 4e-9), (1, 2, 0), 5)]


@pytest.mark.parametrize("n,cell,pbc,acc", NEAR)
def test_near_table_is_bit_exact(mmx, n, cell, pbc, acc):
    plan = mmx.DemagPlan(n, cell, pbc, accuracy=acc, keep_real_kernel=True)
    got = plan.real_kernel()
    K9 = O.kernel_arne(plan.p, cell, pbc, acc)
    assert np.array_equal(got.view(np.uint32), K9[:6].view(np.uint32))


# lines per workgroup 8, 4, 2, 1 and lines that do not fill the last tile
LINES = [(2, 6, 10), (1, 9, 130), (2, 100, 5), (3, 300, 4), (1, 4, 700), (1, 1100, 3), (2, 2048, 2), (40, 3, 4)]


@pytest.mark.parametrize("n", LINES)
def test_octant_is_the_fp64_transform(mmx, n):
    plan = mmx.DemagPlan(n, (3e-9, 4e-9, 4e-9), keep_real_kernel=True)
    real = plan.real_kernel().astype(np.float64)
    got = plan.kernel()
    top = np.abs(real).max()
    ko = plan.ko
    for c in range(6):
        if np.abs(real[c]).max() < 1e-5 * top:
            assert not got[c].any()
            continue
        want = np.fft.rfftn(real[c]).real[:ko[0], :ko[1], :ko[2]] / real[c].size
        # one rounding to float32 of a value below the largest one, with the
        # FP64 transforms' own error (about 1e-15 per stage) far below it
        assert np.abs(got[c] - want).max() <= 2.0 ** -24 * np.abs(want).max() * 1.01
