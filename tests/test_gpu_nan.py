"""A NaN in the torque ends a step with MMX_ERR_NAN on every corrector epilogue
(two cells at a time with uniform parameters or maps, one cell at a time; the
register-FFT, composite-radix and per-prime x passes, and the batch)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ERR_NAN = 6


@pytest.fixture()
def mmx():
    import mmx
    mmx.check(mmx.lib().mmx_init(0))
    yield mmx
    mmx.check(mmx.lib().mmx_set_fast_x_min_blocks(256, None))


def _sim(mmx, n, maps, zl, solver):
    rng = np.random.default_rng(sum(n))
    s = mmx.Sim(n, (3e-9, 4e-9, 4e-9))
    for k, v in (("Msat", 8e5), ("Aex", 1.3e-11), ("alpha", 0.05), ("m_maxerror", 1e-5), ("dt", 1e-15)):
        s.setv(k, v)
    if zl:
        s.load("zhang-li")
        s.setv("j", (0.0, 0.0, 1e12))
    if solver:
        s.load(solver)
    if maps:
        s.setmask("Aex", rng.uniform(0.5, 1.5, n).astype(np.float32))
    return s, rng.standard_normal((3,) + n).astype(np.float32)


# (grid, maps, spin-transfer torque, workgroups from which the register x passes run)
GRIDS = [((11, 100, 24), False, False, 256),    # composite radices, two cells
         ((11, 100, 24), True, False, 256),
         ((11, 100, 24), False, True, 256),     # one cell
         ((4, 16, 32), False, False, 0),        # register FFT, two cells
         ((4, 16, 32), True, False, 0),
         ((4, 16, 32), False, False, 256),      # composite radices, one cell
         ((3, 10, 17), False, False, 256)]      # one stage per prime


@pytest.mark.parametrize("solver", ["", "solver/heun"])
@pytest.mark.parametrize("n,maps,zl,blocks", GRIDS)
def test_nan_cell_is_reported(mmx, n, maps, zl, blocks, solver):
    print("nan", n, maps, zl, blocks, solver, flush=True)
    mmx.check(mmx.lib().mmx_set_fast_x_min_blocks(blocks, None))
    s, m = _sim(mmx, n, maps, zl, solver)
    s.setarray("m", m)
    s.steps(2)              # a finite state steps
    m[1, n[0] - 1, n[1] // 2, 3] = np.nan
    s.setarray("m", m)
    with pytest.raises(mmx.MMXError) as e:
        s.steps(1)
    assert e.value.code == ERR_NAN
    assert s.getv("step") == 2
    m[np.isnan(m)] = 0.5
    s.setarray("m", m)      # the slots are left clear
    s.steps(1)
    assert s.getv("step") == 3


@pytest.mark.parametrize("n,blocks", [((11, 100, 24), 256), ((4, 16, 32), 0), ((4, 16, 32), 256)])
def test_nan_of_a_local_term(mmx, n, blocks):
    """A NaN that enters through the applied field of one cell alone."""
    mmx.check(mmx.lib().mmx_set_fast_x_min_blocks(blocks, None))
    s, m = _sim(mmx, n, False, False, "")
    s.setv("B_ext", (0.01, 0.01, 0.01))
    mask = np.ones((3,) + n, np.float32)
    mask[2, 0, 1, 5] = np.nan
    s.setmask("B_ext", mask, 3)
    s.setarray("m", m)
    with pytest.raises(mmx.MMXError) as e:
        s.steps(1)
    assert e.value.code == ERR_NAN


def test_nan_in_a_batch(mmx):
    good, bad = _sim(mmx, (1, 16, 32), False, False, ""), _sim(mmx, (2, 20, 24), False, False, "")
    bad[1][0, 0, 0, 0] = np.nan
    for s, m in (good, bad):
        s.setarray("m", m)
    with pytest.raises(mmx.MMXError) as e:
        mmx.Batch([good[0], bad[0]]).steps(2)
    assert e.value.code == ERR_NAN
