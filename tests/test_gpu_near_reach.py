"""The reach of the near-field table ends for any cell size that a plan takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a grid of more than 2^20 displacements, on which the reach is shortened until
# the table fits; infinite cells give no finite kernel value: a zero kernel
@pytest.mark.parametrize("cell", [(float("inf"),) * 3, (3e-9, 3e-9, 3e-9)])
def test_reach_ends(cell):
    import mmx
    mmx.check(mmx.lib().mmx_init(0))
    print("reach", cell, flush=True)
    k = mmx.DemagPlan((64, 64, 64), cell).kernel()
    assert np.isfinite(k).all() and k.any() == np.isfinite(cell[0])
