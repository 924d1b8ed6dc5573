"""The GPU tests of the composite-radix passes cover every radix that the plans
can choose (the rule and the lengths are in test_gpu_comp_passes.py)."""
from test_gpu_comp_passes import LARGE_RADIX, LARGE_RADIX_X, _compiled_radices, _radices


def test_every_radix_above_16_is_planned():
    above = {r for r in _compiled_radices() if r > 16}
    assert len(_compiled_radices()) == 27
    assert {r for p in LARGE_RADIX.values() for r in p if r > 16} == above
    # x takes the larger class below 512 points on many rows (plan_init)
    reach = set()
    for Lx in range(1, 512):
        p = _radices(Lx, 32)
        reach |= {r for r in p if r > 16}
    assert {r for p in LARGE_RADIX_X.values() for r in p if r > 16} == reach
