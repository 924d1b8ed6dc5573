"""The composite-radix demag passes at every radix and at the sizes where their
tiles, stages and plans change: B against a float64 FFT of the plan's own
real-space kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mmx():
    import mmx
    mmx.check(mmx.lib().mmx_init(0))
    return mmx


def _check(mmx, n, pbc=(0, 0, 0), masked=False):
    import torch
    print("comp pass", n, pbc, flush=True)
    plan = mmx.DemagPlan(n, (3e-9, 4e-9, 4e-9), pbc, keep_real_kernel=True)
    K = plan.real_kernel().astype(np.float64)
    K[np.abs(K).max(axis=(1, 2, 3)) < 1e-5 * np.abs(K).max()] = 0.0
    rng = np.random.default_rng(1000 * n[0] + 10 * n[1] + n[2])
    m = rng.standard_normal((3,) + n).astype(np.float32)
    ms = rng.uniform(0.0, 2.0, n).astype(np.float32) if masked else None
    dm = torch.from_numpy(m).cuda()
    b = torch.full((3,) + n, np.nan, device="cuda")
    dms = None if ms is None else torch.from_numpy(ms).cuda()
    plan.update_b(b.data_ptr(), dm.data_ptr(), 8e5, None if ms is None else dms.data_ptr(), None)
    torch.cuda.synchronize()
    S = np.fft.rfftn(m.astype(np.float64) * (1.0 if ms is None else ms), s=plan.p, axes=(1, 2, 3))
    kh = np.fft.rfftn(K, axes=(1, 2, 3))
    rows = ((0, 5, 4), (5, 1, 3), (4, 3, 2))
    F = np.stack([sum(kh[rows[c][s]] * S[s] for s in range(3)) for c in range(3)])
    want = np.fft.irfftn(F, s=plan.p, axes=(1, 2, 3))[:, :n[0], :n[1], :n[2]] * (4e-7 * np.pi * 8e5)
    # float32 roundings: some ten per transform, six transforms, and the kernel's own
    assert np.abs(b.cpu().numpy() - want).max() <= 4e-6 * np.abs(want).max()


# x half-lengths: one stage, two and three stages of radices up to 16 (which is
# what few rows take), 25 x 25, primes 11 and 13, odd lengths
X = [3, 7, 9, 11, 13, 15, 18, 20, 21, 22, 25, 26, 27, 28, 30, 33, 39, 42, 44, 45, 50, 60, 63, 65, 66, 75, 77, 78, 81,
     88, 90, 91, 99, 100, 104, 110, 117, 120, 121, 125, 130, 143, 150, 156, 169, 176, 195, 200, 208, 210, 225, 240,
     250, 270, 286, 300, 343, 360, 375, 420, 500, 600, 625, 729, 1000]


@pytest.mark.parametrize("nx", X)
def test_x_lengths(mmx, nx):
    _check(mmx, (1, 3, nx))


@pytest.mark.parametrize("n,pbc", [((9, 240, 20), (0, 0, 0)), ((1, 6, 100), (0, 0, 1)), ((3, 700, 75), (0, 0, 0)),
                                   ((1, 5, 1024), (0, 0, 0)), ((2, 10, 130), (0, 0, 1))])
def test_x_rows(mmx, n, pbc):
    _check(mmx, n, pbc, masked=True)


# y: two and three stages of both classes, columns that do not fill a tile
@pytest.mark.parametrize("ny", [5, 11, 13, 25, 33, 50, 65, 75, 100, 110, 125, 150, 182, 200, 250, 300, 338, 500, 550,
                                625, 750, 1000])
def test_y_lengths(mmx, ny):
    _check(mmx, (2, ny, 5))


@pytest.mark.parametrize("ny,nx,pbc", [(5, 20, 0), (13, 7, 0), (25, 33, 0), (50, 2, 0), (75, 17, 0), (125, 70, 0),
                                       (100, 9, 1), (200, 40, 0), (250, 3, 0), (300, 16, 0), (500, 5, 0),
                                       (600, 4, 0), (750, 6, 0), (1000, 9, 0), (1024, 10, 0), (338, 4, 1)])
def test_film_y_lengths(mmx, ny, nx, pbc):
    _check(mmx, (1, ny, nx), (0, pbc, 0))


# z: every register column length, the lengths behind them, periodic
@pytest.mark.parametrize("nz", list(range(2, 17)) + [18, 20, 22, 25, 26, 27, 33, 36, 50, 60, 75, 110, 125, 250, 300])
def test_z_lengths(mmx, nz):
    _check(mmx, (nz, 4, 9))


@pytest.mark.parametrize("n,pbc", [((10, 6, 30), (1, 0, 0)), ((22, 4, 10), (1, 1, 0)), ((5, 70, 50), (0, 1, 0)),
                                   ((11, 20, 44), (0, 0, 1)), ((36, 10, 40), (0, 0, 0))])
def test_z_grids(mmx, n, pbc):
    _check(mmx, n, pbc, masked=True)


# batches whose passes hold the composite tiles alone, the 64-column z tile
# alone, and generic tiles next to them (primes above 13, a radix above 16)
BATCHES = [[(1, 16, 32), (1, 20, 50)], [(2, 16, 32), (4, 12, 20), (8, 6, 10)], [(9, 8, 16), (2, 16, 32), (1, 30, 21)],
           [(1, 17, 19), (2, 16, 32), (3, 34, 10)], [(1, 250, 4), (20, 4, 6), (1, 625, 2)]]


@pytest.mark.parametrize("grids", BATCHES)
def test_batch_tiles(mmx, grids):
    def make(n, k):
        s = mmx.Sim(n, (3e-9, 4e-9, 4e-9))
        for name, v in (("Msat", 8e5), ("Aex", 1.3e-11), ("alpha", 0.1), ("m_maxerror", 1e-5), ("dt", 1e-14)):
            s.setv(name, v)
        s.load("zhang-li")
        s.setv("j", (0.0, 0.0, 1e12))
        s.setarray("m", np.random.default_rng(k).standard_normal((3,) + n).astype(np.float32))
        return s
    print("batch", grids, flush=True)
    one = [make(n, k) for k, n in enumerate(grids)]
    both = [make(n, k) for k, n in enumerate(grids)]
    mmx.Batch(both).steps(3)
    for a, b in zip(one, both):
        a.steps(3)
        # three steps of float32 stages of the same arithmetic in other transforms
        assert np.abs(a.getarray("m") - b.getarray("m")).max() < 5e-6
        assert a.getv("step") == b.getv("step") == 3


# grids of more rows than workgroups wanted: the two-cell epilogue with uniform
# parameters and with maps, and the per-cell one with the spin-transfer torque,
# on radices up to 16 (above: test_cells_in_pairs_large_radix); the corrector's
# maximum over many workgroups
@pytest.mark.parametrize("maps", [False, True])
@pytest.mark.parametrize("zl", [False, True])
@pytest.mark.parametrize("n,pbc", [((11, 100, 24), (0, 0, 0)), ((2, 650, 22), (0, 0, 1)), ((3, 350, 9), (0, 1, 0))])
def test_cells_in_pairs(mmx, n, pbc, zl, maps):
    from oracle import oracle as O
    print("pairs", n, pbc, zl, maps, flush=True)
    cell = (3e-9, 4e-9, 5e-9)
    rng = np.random.default_rng(n[1])
    sim = mmx.Sim(n, cell, pbc)
    kw = dict(msat=8e5, aex=1.3e-11, alpha=0.05, bext=(0.01, 0.0, 0.02), ku=4e5, anis_u=(0.6, 0.0, 0.8))
    for k, v in (("Msat", 8e5), ("Aex", 1.3e-11), ("alpha", 0.05), ("B_ext", kw["bext"])):
        sim.setv(k, v)
    sim.load("anisotropy/uniaxial")
    sim.setv("Ku", 4e5)
    sim.setv("anisU", (0.6, 0.0, 0.8))
    if zl:
        sim.load("zhang-li")
        sim.setv("j", (2e11, 0.0, 1e12))
        sim.setv("polarisation", 0.56)
        sim.setv("xi", 0.05)
        kw.update(j=(2e11, 0.0, 1e12), pol=0.56, xi=0.05)
    if maps:
        ms = rng.uniform(0.5, 1.0, n).astype(np.float32)
        ax = rng.uniform(0.5, 1.5, n).astype(np.float32)
        sim.setmask("Msat", ms)
        sim.setmask("Aex", ax)
        kw.update(msat_map=ms, aex_map=ax)
    m = rng.standard_normal((3,) + n).astype(np.float32)
    sim.setarray("m", m)
    prob = O.Problem(n, cell, pbc=pbc, **kw)
    mo = prob.normalized(m.astype(np.float64))
    want = prob.heff(mo)
    # the repository's parity bar for fields, relative to the largest value
    assert np.abs(sim.getarray("H_eff") - want).max() <= 1e-5 * np.abs(want).max()
    e_gpu, e_orc = sim.try_step(1e-15), prob.try_step(mo, 1e-15)
    assert abs(e_gpu - e_orc) <= 1e-4 * e_orc
    assert np.abs(sim.getarray("m") - prob.normalized(mo)).max() <= 1e-5


# the class of radices above 16: every one of them in y, in a film's y and in z,
# and those that x uses on grids of more than 2048 rows
LARGE_RADIX = {324: (18, 18), 400: (20, 20), 294: (21, 14), 484: (22, 22), 768: (32, 24), 350: (25, 14),
               676: (26, 26), 594: (27, 22), 784: (28, 28), 900: (30, 30)}
LARGE_RADIX_X = {162: (18, 9), 200: (20, 10), 147: (21, 7), 242: (22, 11), 312: (24, 13), 125: (25, 5),
                 338: (26, 13), 243: (27, 9), 392: (28, 14)}


def _radices(L, top2):
    """The rule of comp_plan (comp_x.hip) over the radices of comp_fft.hpp: two
    stages, else three, with the smallest largest radix."""
    have = _compiled_radices()
    two = [(L // r1, r1) for r1 in range(1, top2 + 1)
           if L % r1 == 0 and r1 <= L // r1 <= top2 and {r1, L // r1} <= have]
    if two:
        return min(two)
    three = [(L // r1 // r2, r1, r2) for r2 in range(2, 33) for r1 in range(r2, 33)
             if L % (r1 * r2) == 0 and L // r1 // r2 >= r1 and {r1, r2, L // r1 // r2} <= have]
    return min(three) if three else ()


def _compiled_radices():
    import os
    import re
    src = open(os.path.join(os.path.dirname(__file__), "..", "2_amd", "csrc", "comp_fft.hpp")).read()
    lists = re.findall(r"#define MMX_COMP_RADICES_\d+\(X\)[^\n]*\n([^\n]*)", src)
    return {int(r) for text in lists for r in re.findall(r"X\((\d+)\)", text)}


@pytest.mark.parametrize("L", sorted(LARGE_RADIX))
@pytest.mark.parametrize("axis", ["y", "film", "z"])
def test_large_radices(mmx, L, axis):
    assert _radices(L, 32) == LARGE_RADIX[L]
    k = L // 2
    _check(mmx, {"y": (2, k, 5), "film": (1, k, 5), "z": (k, 3, 5)}[axis])


@pytest.mark.parametrize("Lx", sorted(LARGE_RADIX_X))
def test_large_radices_x(mmx, Lx):
    assert _radices(Lx, 32) == LARGE_RADIX_X[Lx]
    _check(mmx, (1, 2100, 2 * Lx), (0, 1, 1))


# the epilogues in the larger class: fields, first stage and corrector
@pytest.mark.parametrize("maps", [False, True])
@pytest.mark.parametrize("zl", [False, True])
def test_cells_in_pairs_large_radix(mmx, zl, maps):
    n = (3, 700, 162)
    assert _radices(n[2], 32) == (18, 9) and n[0] * n[1] > 2048
    test_cells_in_pairs(mmx, n, (0, 0, 0), zl, maps)


# arrays that start off an 8-byte boundary take one cell at a time: the same bits
@pytest.mark.parametrize("n", [(2, 520, 20), (1, 6, 100)])
def test_arrays_off_the_pair_boundary(mmx, n):
    import torch
    print("unaligned", n, flush=True)
    plan = mmx.DemagPlan(n, (3e-9, 4e-9, 4e-9))
    rng = np.random.default_rng(n[1])
    N = int(np.prod(n))
    src = [rng.standard_normal(3 * N).astype(np.float32), rng.uniform(0.5, 1.5, N).astype(np.float32)]

    def field(om, ob, os_):
        m, s = (torch.zeros(a.size + 2, device="cuda") for a in src)
        b = torch.full((3 * N + 2,), np.nan, device="cuda")
        m[om:om + 3 * N] = torch.from_numpy(src[0]).cuda()
        s[os_:os_ + N] = torch.from_numpy(src[1]).cuda()
        assert m.data_ptr() % 8 == b.data_ptr() % 8 == s.data_ptr() % 8 == 0
        plan.update_b(b.data_ptr() + 4 * ob, m.data_ptr() + 4 * om, 8e5, s.data_ptr() + 4 * os_, None)
        torch.cuda.synchronize()
        out = b.cpu().numpy()
        assert np.isnan(out[:ob]).all() and np.isnan(out[ob + 3 * N:]).all()
        return out[ob:ob + 3 * N]
    want = field(0, 0, 0)
    assert np.isfinite(want).all()
    for off in ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)):
        assert np.array_equal(field(*off), want)
