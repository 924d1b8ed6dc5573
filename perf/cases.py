"""Performance cases of the solver core: what is timed, and the same results in 64 bits.

A case is one pass of work through the package's public entry points, on data
that is resident on the GPU, as a simulation script has it:

    steps   Sim.steps(count) with solver/rk12 (adaptive) or solver/heun, then
            the table's <m>; returns m and <m>
    field   Sim.update of H_eff or of the torque at a new m; returns the field
    batch   Batch.steps(count) of uneven films; returns every m
    plan    construction of a demag plan and its first field
    kernels one field evaluation and RK stage composed from the drop-in
            kernels, as an engine on the C entry points composes it
    train   one training step of the learned demag correction; returns the
            loss and the gradients

Sizes are the user's (x, y, z) cells; arrays are in internal (z, y, x) order.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "2_amd"))

import mmx  # noqa: E402
from mmx import kernels  # noqa: E402

MU0 = 4.0 * math.pi * 1e-7
GAMMA = 2.211e5
MU_B, Q_E = 9.2740091523e-24, 1.60217646e-19
AEX = 1.3e-11
J_X = 1e12      # A/m^2, with the Zhang-Li torque
POL, XI = 0.56, 0.05

BASE = {"kind": "steps", "nx": 0, "ny": 0, "nz": 1, "cell": 4.0, "cellz": 3.0, "msat": 8e5, "alpha": 0.02,
        "ku": 0.0, "bext": 0.0, "pbc_x": 0, "pbc_y": 0, "pbc_z": 0, "disk": False, "aex_map": False,
        "zl": False, "temp": 0.0, "solver": "rk12", "dt": 2e-14, "count": 1, "quantity": "H_eff"}


def _case(**kw):
    return {**BASE, **kw}


def listed():
    return [
        # the standard-problem film: the smallest grid people run, bound by launches and latency
        _case(name="film_128x32x1_rk12", nx=128, ny=32, cell=3.90625, bext=0.01, count=20),
        # a film on round decimal sizes (500 nm x 125 nm) under a spin-polarised current: lengths with factors of 5
        _case(name="film_500x125x1_zhangli_rk12", nx=500, ny=125, cell=1.0, cellz=3.0, zl=True, count=10),
        # what every script waits for first: the demag kernel of its grid, up to the first field
        _case(name="plan_200x200x5_first_field", kind="plan", nx=200, ny=200, nz=5),
        # ragged, periodic along x, patterned (geometry mask and exchange map): the torque for a relaxation check
        _case(name="ragged_96x70x11_torque", kind="field", nx=96, ny=70, nz=11, pbc_x=1, disk=True, aex_map=True,
              quantity="torque"),
        # a patterned disk at 300 K: fixed-step Heun, a new thermal field in each step
        _case(name="disk_200x200x5_thermal_heun", nx=200, ny=200, nz=5, disk=True, temp=300.0, solver="heun",
              dt=1e-14, count=10),
        # the headline grid: one field evaluation, and adaptive steps
        _case(name="bulk_256x256x64_field", kind="field", nx=256, ny=256, nz=64, cellz=4.0, ku=5e5, alpha=0.1),
        _case(name="bulk_256x256x64_rk12", nx=256, ny=256, nz=64, cellz=4.0, ku=5e5, alpha=0.1, count=4),
        # a wide film, one layer
        _case(name="film_1024x1024x1_field", kind="field", nx=1024, ny=1024, cell=5.0, cellz=5.0),
        # the largest grid: a thick film with long rows
        _case(name="film_1024x1024x32_field", kind="field", nx=1024, ny=1024, nz=32, cell=2.0, cellz=2.0, msat=1e6),
        # a parameter study: uneven films stepped together
        _case(name="batch_32_films_rk12", kind="batch", films=32, cell=4.0, cellz=3.0, zl=True, count=8),
        # an engine of its own on the drop-in kernels and the demag plan
        _case(name="kernels_240x200x36", kind="kernels", nx=240, ny=200, nz=36, cellz=4.0, ku=5e5, bext=0.01,
              zl=True, disk=True, alpha=0.1),
        # learned demag correction: training on exact fields
        _case(name="surrogate_256x256x4_train", kind="train", nx=256, ny=256, nz=4),
    ]


def _smooth(rng, lo, hi, even=False):
    """A size spread over the logarithm of [lo, hi] whose primes are at most 13 (sizes that scripts use)."""
    while True:
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        r = n
        for p in (2, 3, 5, 7, 11, 13):
            while r % p == 0:
                r //= p
        if r == 1 and lo <= n <= hi and not (even and n % 2):
            return n


def draw(rng):
    kind = rng.choices(("steps", "field", "plan", "kernels", "batch", "train"), (42, 28, 8, 9, 8, 5))[0]
    c = _case(kind=kind, cell=rng.choice((1.0, 2.0, 2.5, 4.0, 5.0)), cellz=rng.choice((2.0, 3.0, 4.0)),
              msat=round(rng.uniform(6e5, 1.2e6)), alpha=round(rng.uniform(0.01, 0.2), 4))
    if kind == "batch":
        c.update(films=rng.randint(8, 48), zl=True, cell=4.0, cellz=3.0, count=rng.randint(4, 12))
        return c
    if kind == "train":
        c.update(nx=16 * rng.randint(4, 16), ny=16 * rng.randint(4, 16), nz=rng.randint(1, 5), cell=4.0)
        return c
    most = {"field": 1 << 23, "plan": 200000}.get(kind, 1 << 22)
    while True:
        nx, ny = _smooth(rng, 16, 1024, even=True), _smooth(rng, 16, 1024, even=True)
        nz = 1 if rng.random() < 0.35 else _smooth(rng, 2, 64)
        if nx * ny * nz <= most and max(nx, ny) <= 32 * min(nx, ny):
            break
    c.update(nx=nx, ny=ny, nz=nz, ku=rng.choice((0.0, 0.0, 5e5)), bext=rng.choice((0.0, 0.01, 0.05)),
             disk=rng.random() < 0.3, zl=rng.random() < 0.3)
    if rng.random() < 0.25:
        c[rng.choice(("pbc_x", "pbc_y"))] = 1
    if kind == "plan":
        c.update(cell=4.0, cellz=rng.choice((3.0, 4.0)), ku=0.0, bext=0.0, disk=False, zl=False, pbc_x=0, pbc_y=0)
    if kind == "field":
        c.update(quantity=rng.choice(("H_eff", "H_eff", "torque")), aex_map=rng.random() < 0.2)
    if kind == "steps":
        c["count"] = max(1, min(20, (1 << 23) // (nx * ny * nz)))
        if rng.random() < 0.3:
            c.update(solver="heun", dt=1e-14, temp=rng.choice((0.0, 300.0)), zl=False)
    return c


# ------------------------------------------------------------------ inputs

def _n(case):
    return case["nz"], case["ny"], case["nx"]


def _cell(case):
    return case["cellz"] * 1e-9, case["cell"] * 1e-9, case["cell"] * 1e-9


def _pbc(case):
    return case["pbc_z"], case["pbc_y"], case["pbc_x"]


def _texture(n, seed):
    """A smooth unit field with some short-range disorder (float32, on the GPU): long waves along each axis
    around a mean direction, as a state under way has them, made from the seed alone."""
    r = random.Random(seed)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = [torch.arange(k, device="cuda", dtype=torch.float32) / k for k in n]
    m = torch.empty((3,) + tuple(n), device="cuda", dtype=torch.float32)
    for c in range(3):
        m[c] = r.uniform(0.3, 0.8)
        for _ in range(6):
            k = [r.randint(0, 3) for _ in range(3)]
            ph = [2 * math.pi * k[a] * x[a] + r.uniform(0, 6.28) for a in range(3)]
            m[c] += r.uniform(0.2, 0.6) * (torch.sin(ph[0])[:, None, None] * torch.sin(ph[1])[None, :, None]
                                           * torch.sin(ph[2])[None, None, :])
    m += 0.05 * torch.randn(m.shape, device="cuda", generator=g)
    m /= torch.linalg.vector_norm(m.double(), dim=0).float()
    return m


def _disk(n):
    """1 inside the ellipse that fills the film plane, 0 outside."""
    y = (torch.arange(n[1], device="cuda", dtype=torch.float64) + 0.5) / n[1] * 2 - 1
    x = (torch.arange(n[2], device="cuda", dtype=torch.float64) + 0.5) / n[2] * 2 - 1
    return ((y * y)[:, None] + (x * x)[None, :] <= 1.0).float().expand(n).contiguous()


def _aex_map(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 77)
    return 0.5 + torch.rand(n, device="cuda", generator=g)


def _bext(case):
    """An applied field in the film plane (internal order), tesla."""
    return 0.0, 0.3 * case["bext"], case["bext"]


def _films(case, seed):
    """The films of a batch: 32x32x1 .. 256x128x4 cells, each with its own Ms and damping."""
    r = random.Random(1000 + case["films"])
    out = []
    for i in range(case["films"]):
        out.append({**case, "kind": "steps", "nx": 32 * r.randint(1, 8), "ny": 32 * r.randint(1, 4),
                    "nz": r.randint(1, 4), "msat": round(r.uniform(6e5, 1.2e6)),
                    "alpha": round(r.uniform(0.005, 0.1), 4), "seed": seed * 1000 + i})
    return out


class _Floats:
    """Device floats of a simulation as a tensor's source; keeps the simulation alive."""

    def __init__(self, sim, ptr):
        self.sim = sim
        self.__cuda_array_interface__ = {"shape": (3,) + sim.n, "typestr": "<f4", "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(sim, name):
    return torch.as_tensor(_Floats(sim, sim.device_array(name)), device="cuda")


def _sim(case, seed):
    n = _n(case)
    s = mmx.Sim(n, _cell(case), _pbc(case))
    s.setv("Msat", case["msat"])
    s.setv("Aex", AEX)
    s.setv("alpha", case["alpha"])
    s.setv("gamma", GAMMA)
    s.setv("B_ext", _bext(case))
    s.setv("m_maxerror", 1e-5)
    if case["ku"]:
        s.load("anisotropy/uniaxial")
        s.setv("Ku", case["ku"])
        s.setv("anisU", (1.0, 0.0, 0.0))
    if case["zl"]:
        s.load("zhang-li")
        s.setv("j", (0.0, 0.0, J_X))
        s.setv("polarisation", POL)
        s.setv("xi", XI)
    if case["solver"] != "rk12":
        s.load("solver/" + case["solver"])
    if case["temp"]:
        s.load("temperature/brown")
        s.setv("Temp", case["temp"])
        s.setv("Therm_seed", seed)
    if case["disk"]:
        s.setmask("Msat", _disk(n).cpu().numpy())
    if case["aex_map"]:
        s.setmask("Aex", _aex_map(n, seed).cpu().numpy())
    s.setv("dt", case["dt"])
    _view(s, "m").copy_(_texture(n, seed))
    torch.cuda.synchronize()
    s.update("m")
    return s


def prepare(case, seed):
    mmx.check(mmx.lib().mmx_init(0))
    if case["kind"] == "batch":
        sims = [_sim(c, c["seed"]) for c in _films(case, seed)]
        return {"case": case, "sims": sims, "batch": mmx.Batch(sims)}
    if case["kind"] == "plan":
        m = _texture(_n(case), seed)
        return {"case": case, "m": m, "b": torch.zeros_like(m)}
    if case["kind"] == "kernels":
        n = _n(case)
        z = lambda: torch.zeros((3,) + n, device="cuda")  # noqa: E731
        msat = _disk(n) if case["disk"] else None
        m = _texture(n, seed)
        if msat is not None:
            m *= msat
        return {"case": case, "plan": mmx.DemagPlan(n, _cell(case), _pbc(case)), "m": m, "msat": msat,
                "red": mmx.Reductor(3 * m[0].numel()), "b": z(), "h": z(), "w": z(), "tau": z(), "m1": z()}
    s = _sim(case, seed)
    if case["kind"] == "train":
        return {"case": case, "sim": s, "sur": mmx.Surrogate(s, seed=seed), "m": _view(s, "m").clone()}
    if case["kind"] == "field":
        s.update(case["quantity"])      # builds the demag plan
        return {"case": case, "sim": s, "out": _view(s, "H_eff" if case["quantity"] == "H_eff" else "torque")}
    s.update("H_eff")
    return {"case": case, "sim": s}


# ---------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "steps":
        s = state["sim"]
        s.steps(case["count"])
        avg = s.getv("<m>")
        return {"m": _view(s, "m"), "avg": np.array(avg, dtype=np.float32)}
    if kind == "field":
        state["sim"].update(case["quantity"])
        return {case["quantity"]: state["out"]}
    if kind == "plan":
        plan = mmx.DemagPlan(_n(case), _cell(case), _pbc(case))
        plan.update_b(state["b"].data_ptr(), state["m"].data_ptr(), case["msat"], None,
                      torch.cuda.current_stream().cuda_stream)
        return {"B": state["b"]}
    if kind == "batch":
        state["batch"].steps(case["count"])
        return {"m": [_view(s, "m") for s in state["sims"]]}
    if kind == "train":
        loss = state["sur"].train_step(state["m"].data_ptr(), 5e-4)
        return {"loss": np.array([loss], dtype=np.float32), "grads": state["sur"].get_grads()}
    # the engine's sum of field terms, torque terms and the predictor
    m, msat, h, w, tau, m1 = (state[k] for k in ("m", "msat", "h", "w", "tau", "m1"))
    cell, pbc, ms = _cell(case), _pbc(case), case["msat"]
    st = torch.cuda.current_stream().cuda_stream
    state["plan"].update_b(state["b"].data_ptr(), m.data_ptr(), ms, None if msat is None else msat.data_ptr(), st)
    kernels.exchange6(m, 2 * AEX / (MU0 * ms), cell, pbc, msat_map=msat, out=h)
    kernels.vec_madd(h, state["b"], (1 / MU0,) * 3, out=h)
    if case["ku"]:
        kernels.uniaxial_anisotropy(m, 2 * case["ku"] / (MU0 * ms), (1.0, 0.0, 0.0), msat_map=msat, out=w)
        kernels.vec_madd(h, w, (1.0, 1.0, 1.0), out=h)
    kernels.vec_madd(h, None, tuple(b / MU0 for b in _bext(case)), out=h)
    kernels.torque(m, h, case["alpha"], out=tau)
    if case["zl"]:
        kernels.zhangli(m, (0.0, 0.0, J_X), POL * MU_B / (Q_E * ms), XI, case["alpha"], cell, pbc, msat_map=msat,
                        out=w)
        kernels.vec_madd(tau, w, (1 / GAMMA,) * 3, out=tau)
    kernels.madd(m, tau, case["dt"] * GAMMA, out=m1)
    kernels.normalize(m1, msat)
    top = state["red"].maxnorm(tau[0].data_ptr(), tau[1].data_ptr(), tau[2].data_ptr(), tau[0].numel(), st)
    return {"H_eff": h, "torque": tau, "m1": m1, "maxtorque": np.array([top], dtype=np.float32)}


# -------------------------------------------------------- what it must cost

def _eval_work(case):
    """(bytes of the field's own data: m in, field out, kernel octant in; flops of one zero-padded convolution
    with the local terms): real transforms of the rows that hold data, complex ones along y and z, there and
    back, three components."""
    n = _n(case)
    p = [k if k == 1 or b else 2 * k for k, b in zip(n, _pbc(case))]
    cells, h2 = n[0] * n[1] * n[2], p[2] // 2 + 1
    lg = lambda k: math.log2(k) if k > 1 else 0.0  # noqa: E731
    fft = 2.5 * n[0] * n[1] * p[2] * lg(p[2]) + 5.0 * n[0] * h2 * p[1] * lg(p[1]) + 5.0 * p[1] * h2 * p[0] * lg(p[0])
    octant = 24.0 * (p[0] // 2 + 1) * (p[1] // 2 + 1) * h2
    return 24.0 * cells + octant, 6 * fft + 30.0 * p[0] * p[1] * h2 + 80.0 * cells


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_eval_work(c) for c in _films(case, 0)]
        return {"bytes": sum(b for b, _ in each) * case["count"], "flops": sum(f for _, f in each) * 2 * case["count"]}
    b, f = _eval_work(case)
    cells = _n(case)[0] * _n(case)[1] * _n(case)[2]
    if kind == "steps":
        return {"bytes": b * case["count"], "flops": f * 2 * case["count"]}
    if kind == "field":
        return {"bytes": b + (4.0 * cells if case["disk"] else 0) + (4.0 * cells if case["aex_map"] else 0), "flops": f}
    if kind == "plan":      # per displacement and source axis: 4 points' pairs of poles at least, in 64 bits
        return {"bytes": b, "flops": f + 3 * 4 * 50.0 * 8 * cells}
    if kind == "kernels":   # m and the mask in; H_eff, torque and the predictor out
        return {"bytes": b + 28.0 * cells, "flops": f + 120.0 * cells}
    pixels = case["nx"] * case["ny"]    # forward, backward-data and weight gradients of four 3x3 layers
    conv = 2.0 * 9 * pixels * (3 * 32 * 32 + 32 * 16)
    return {"bytes": b + 8.0 * 32297, "flops": f + 3 * conv}


# ------------------------------------------------- the same method in 64 bits

def _dipole_octant(ext, cell, accuracy=6):
    """Six components (zz-order 00,11,22,12,02,01 of the internal axes) of the cell-averaged dipole kernel at the
    displacements 0..ext-1 per axis: surface charges of the source cell on its two faces, averaged over the points
    of the destination cell, point counts by distance."""
    dev, f8 = "cuda", torch.float64
    g = torch.meshgrid(*[torch.arange(e, device=dev, dtype=f8) for e in ext], indexing="ij")
    d = [torch.clamp(a - 1, min=0) * c for a, c in zip(g, cell)]
    dist = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2).reshape(-1)
    dist[dist == 0] = min(cell)
    # divisions by tensors: by a number they are products with its inverse, and the point counts jump where the
    # quotient is a half
    size = dist / torch.full_like(dist, accuracy)
    num = torch.stack([(torch.clamp(torch.full_like(size, c) / size, min=1.0) + 0.5).to(torch.int64) for c in cell])
    R = [a.reshape(-1) * c for a, c in zip(g, cell)]
    key = (num[0] * 4096 + num[1]) * 4096 + num[2]
    out = torch.zeros(6, dist.numel(), device=dev, dtype=f8)
    pick = {(0, 0): 0, (1, 1): 1, (2, 2): 2, (1, 2): 3, (0, 2): 4, (0, 1): 5}
    for k in torch.unique(key).tolist():
        sel = (key == k).nonzero().reshape(-1)
        q = [k >> 24, (k >> 12) & 4095, k & 4095]
        off = [((torch.arange(q[a], device=dev, dtype=f8) + 0.5) / q[a] - 0.5) * cell[a] for a in range(3)]
        for s in range(3):
            v, w = (s + 1) % 3, (s + 2) % 3
            face = {v: ((torch.arange(2 * q[v], device=dev, dtype=f8) + 0.5) / (2 * q[v]) - 0.5) * cell[v],
                    w: ((torch.arange(2 * q[w], device=dev, dtype=f8) + 0.5) / (2 * q[w]) - 0.5) * cell[w]}
            # destination points minus face points along each axis
            sep = [off[s] if a == s else (off[a][:, None] - face[a][None, :]).reshape(-1) for a in range(3)]
            npts = sep[0].numel() * sep[1].numel() * sep[2].numel()
            charge = cell[v] * cell[w] / npts
            lines = torch.cartesian_prod(*sep)
            step = max(1, (1 << 24) // lines.shape[0])
            for at in range(0, sel.numel(), step):
                i = sel[at:at + step]
                acc = [0.0, 0.0, 0.0]
                for sign in (1.0, -1.0):
                    r = [R[a][i][:, None] + lines[None, :, a] - (sign * cell[s] / 2 if a == s else 0.0)
                         for a in range(3)]
                    f = sign * charge / (4 * math.pi) * (r[0] ** 2 + r[1] ** 2 + r[2] ** 2) ** -1.5
                    for a in range(3):
                        acc[a] = acc[a] + (r[a] * f).sum(1)
                for a in range(s, 3):
                    out[pick[(s, a)], i] = acc[a]
    out = out.reshape((6,) + tuple(ext))
    for (a, b), c in pick.items():
        if a != b:      # odd in both of its axes
            out[c].select(a, 0).zero_()
            out[c].select(b, 0).zero_()
    return out


_PAIR = ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))


def _khat(n, cell, pbc):
    """The six transformed components (real) on the padded grid, and its size."""
    p = [k if k == 1 or b else 2 * k for k, b in zip(n, pbc)]
    most = [(k // 2 - 1) * (b + 1) if k > 1 else 0 for k, b in zip(p, pbc)]
    octant = _dipole_octant([a + 1 for a in most], cell)
    out = []
    for c, (sa, sb) in enumerate(_PAIR):
        k = octant[c]
        for a in range(3):
            if most[a] == 0:
                if p[a] > 1:
                    k = torch.cat([k] + [torch.zeros_like(k)] * (p[a] - 1), dim=a)
                continue
            odd = (sa == a) != (sb == a)
            rest = k.narrow(a, 1, most[a])
            full = torch.cat([torch.flip(rest, (a,)) * (-1.0 if odd else 1.0), k], dim=a)
            at = torch.arange(-most[a], most[a] + 1, device=k.device) % p[a]
            shape = list(k.shape)
            shape[a] = p[a]
            k = torch.zeros(shape, device=k.device, dtype=k.dtype).index_add_(a, at, full)
        out.append(torch.fft.rfftn(k).real.clone())
    return out, p


class _Exact:
    """The same simulation in float64 on plain tensors."""

    def __init__(self, case, seed):
        self.case, self.n, self.cell, self.pbc = case, _n(case), _cell(case), _pbc(case)
        self.khat, self.p = _khat(self.n, self.cell, self.pbc)
        self.ms = case["msat"]
        self.mask = _disk(self.n).double() if case["disk"] else None
        self.aex = _aex_map(self.n, seed).double() if case["aex_map"] else None
        self.m = self.unit(_texture(self.n, seed).double())
        self.t, self.dt = 0.0, case["dt"]

    def unit(self, m):
        r = torch.linalg.vector_norm(m, dim=0)
        m = torch.where(r == 0, torch.zeros_like(m), m / torch.where(r == 0, torch.ones_like(r), r))
        return m if self.mask is None else m * (self.mask != 0)

    def demag(self, m):
        src = m if self.mask is None else m * self.mask
        s = [torch.fft.rfftn(src[c], s=self.p) for c in range(3)]
        k = self.khat
        rows = ((0, 5, 4), (5, 1, 3), (4, 3, 2))
        out = torch.empty_like(m)
        for c in range(3):
            f = k[rows[c][0]] * s[0]
            f += k[rows[c][1]] * s[1]
            f += k[rows[c][2]] * s[2]
            out[c] = torch.fft.irfftn(f, s=self.p)[:self.n[0], :self.n[1], :self.n[2]]
        return self.ms * out

    def side(self, f, axis, by):
        """f one cell further along an axis (of the last three): wrapped, or the edge cell again."""
        a = f.dim() - 3 + axis
        k = f.shape[a]
        at = torch.arange(k, device=f.device) + by
        at = at % k if self.pbc[axis] else at.clamp(0, k - 1)
        return f.index_select(a, at)

    def exchange(self, m):
        out = torch.zeros_like(m)
        lex = None
        if self.mask is not None or self.aex is not None:
            one = torch.ones(self.n, device=m.device, dtype=m.dtype)
            a, s = (one if v is None else v for v in (self.aex, self.mask))
            lex = torch.where(s == 0, torch.zeros_like(s), a / torch.where(s == 0, one, s))
        for axis in range(3):
            for by in (-1, 1):
                d = self.side(m, axis, by) - m
                if lex is not None:
                    o = self.side(lex, axis, by)
                    q = lex + o
                    d = d * torch.where(q == 0, torch.zeros_like(q), 2 * lex * o / torch.where(q == 0, 1 + q, q))
                out += d / self.cell[axis] ** 2
        return 2 * AEX / (MU0 * self.ms) * out

    def field(self, m):
        h = self.demag(m) + self.exchange(m)
        for c, b in enumerate(_bext(self.case)):
            h[c] += b / MU0
        if self.case["ku"]:
            k = 2 * self.case["ku"] / (MU0 * self.ms)
            h[0] += m[0] * (k if self.mask is None else k / torch.where(self.mask == 0, 1 + self.mask, self.mask))
        return h

    def zhangli(self, m):
        """The spin-transfer torque for a current along x; a stencil point outside reads the cell itself."""
        k = m.shape[3]
        at = torch.arange(k, device=m.device)

        def off(by):
            i = at + by
            i = i % k if self.pbc[2] else torch.where((i < 0) | (i >= k), at, i)
            return m.index_select(3, i)

        grad = (off(-2) - 8 * off(-1) + 8 * off(1) - off(2)) / (12 * self.cell[2])
        a = self.case["alpha"]
        coef = J_X * POL * MU_B / (Q_E * self.ms) / ((1 + XI * XI) * (1 + a * a))
        g = -torch.linalg.cross(grad, m, dim=0)
        mg = -torch.linalg.cross(m, g, dim=0)
        out = coef * ((1 + XI * a) * mg + (XI - a) * g)
        if self.mask is not None:
            inv = torch.where(self.mask == 0, torch.zeros_like(self.mask), 1 / torch.where(self.mask == 0, 1 + self.mask, self.mask))
            out = out * inv
        return out

    def torque(self, m, h=None):
        h = self.field(m) if h is None else h
        a = self.case["alpha"]
        x = torch.linalg.cross(m, h, dim=0)
        t = (x - a * torch.linalg.cross(m, x, dim=0)) / (1 + a * a)
        return t + self.zhangli(m) / GAMMA if self.case["zl"] else t

    def attempt(self, t0):
        g = self.dt * GAMMA
        m1 = self.unit(self.m + g * t0)
        t1 = self.torque(m1)
        return self.unit(m1 + 0.5 * g * (t1 - t0)), float((t1 - t0).abs().max()) * g

    def step(self):
        t0 = self.torque(self.m)
        if self.case["solver"] == "heun":
            self.m = self.attempt(t0)[0]
            return
        while True:     # the adaptive rule: headroom 0.8, growth in [0.1, 1.5], smallest step 1 fs
            m, err = self.attempt(t0)
            bad = err > 1e-5
            by = 0.8 * ((1e-5 / err) ** (1.0 / 3.0) if bad else math.sqrt(1e-5 / err))
            self.dt = max(1e-15, self.dt * min(1.5, max(0.1, by)))
            if not bad or self.dt == 1e-15:
                break
        self.m = m


def exact(case, seed):
    kind = case["kind"]
    if kind == "train" or case["temp"]:     # bf16 layers by design; a random field of its own
        return None
    if kind == "batch":
        out = []
        for c in _films(case, seed):
            e = _Exact(c, c["seed"])
            for _ in range(case["count"]):
                e.step()
            out.append(e.m)
        return {"m": out}
    e = _Exact(case, seed)
    if kind in ("plan", "kernels"):     # m as it is given, not normalised first
        e.m = _texture(e.n, seed).double() * (1.0 if e.mask is None else e.mask)
    if kind == "plan":
        return {"B": MU0 * e.demag(e.m)}
    if kind == "steps":
        for _ in range(case["count"]):
            e.step()
        return {"m": e.m, "avg": e.m.reshape(3, -1).mean(1).cpu().numpy()}
    h = e.field(e.m)
    if kind == "field":
        return {case["quantity"]: h if case["quantity"] == "H_eff" else e.torque(e.m, h)}
    tau = e.torque(e.m, h)
    return {"H_eff": h, "torque": tau, "m1": e.unit(e.m + case["dt"] * GAMMA * tau),
            "maxtorque": torch.linalg.vector_norm(tau, dim=0).max().reshape(1).cpu().numpy()}
