"""What a user has this framework do, as measurable cases: time steps of single domains with their
readout (moments, time averages, restart records), ensembles, one tile of a tiled domain, and
gradients by the adjoint.

A case is a dict of plain values, ``prepare`` makes from a seed what a user's program holds before
the call, ``run`` is one pass through the public entry points, ``work`` is what a pass cannot do
without, and ``exact`` is the same pass in 64 bits, written with torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from lbm_amd.domain import BND_HALO, PART_EDGE, PART_INNER, Domain, Ensemble
from lbm_amd.torch_adjoint import ForcingProblem, LatticeKE

SMAGORINSKY = 0.16733      # Vreman constant 2.5 * 0.16733^2 = 0.07
ITURB = 10                 # slice of the inflow-turbulence forcing
AMPL = 1e-3                # its amplitude
NTURB = 50                 # its time slices
UINI = 0.05                # inflow speed
TURBINE_LENGTH, TURBINE_VEL = 4.0, 256.0   # metres per cell, m/s per lattice speed: rotor radius 16 cells

FLOW = dict(kind="flow", q=27, storage="f32", model="reg", ibnd=1, jbnd=0, kbnd=12, kinevisc=1e-3, cylinder=False,
            turbulence=False, turbines=0, readout="moments")


def _flow(name, dims, steps, **kw):
    c = dict(FLOW, nx=dims[0], ny=dims[1], nz=dims[2], steps=steps, **kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a restart record read, a short run, the record written: the smallest grid anybody runs, where launches and
        # latency are all of the time (cylinder in an inflow with turbulence forcing)
        _flow("small_wake_restart", (60, 14, 5), 100, kinevisc=1e-4, cylinder=True, turbulence=True, readout="restart"),
        # plane channel with the plain collision: one closed axis, everything else periodic
        _flow("bgk_channel", (128, 64, 64), 200, q=19, model="bgk", ibnd=0, kbnd=11, kinevisc=1.0 / 30.0),
        # closed box, every wall of its own kind, no size a multiple of anything
        _flow("closed_box", (101, 61, 45), 100, ibnd=22, jbnd=11, kbnd=12),
        # the headline workload: cylinder wake on 9.4 M cells, moments every 200 steps
        _flow("wake_f32", (384, 192, 128), 200, kinevisc=1e-4, cylinder=True, turbulence=True),
        # the same physics in half-precision storage, rows that are no multiple of a wavefront
        _flow("wake_f16", (400, 200, 100), 200, storage="f16s", cylinder=True, turbulence=True),
        # turbulence statistics in double precision: time averages of a sampling window
        _flow("statistics_f64", (150, 90, 70), 100, storage="f64", cylinder=True, turbulence=True, readout="averages"),
        # duct: inflow and four walls
        _flow("duct_f32", (250, 98, 70), 100, jbnd=11, kbnd=11, turbulence=True),
        # wind farm: two rotors, the inflow turbulence drawn anew for every window, time averages
        _flow("wind_farm", (192, 96, 96), 100, kinevisc=1e-4, turbines=2, turbulence=True, readout="averages"),
        # an ensemble of ordinary members, and one of many small ones
        dict(name="ensemble", kind="ensemble", members=16, ni=128, nj=96, nk=80, steps=200, storage="f32"),
        dict(name="ensemble_small", kind="ensemble", members=64, ni=32, nj=24, nk=20, steps=300, storage="f32"),
        # one evaluation and gradient of the forcing problem
        dict(name="adjoint", kind="adjoint", nx=192, ny=96, nz=96, steps=100, every=10, storage="f32"),
        # one GPU's tile of the headline domain (1/8 along j), split steps with the halo transfer between them
        dict(name="tile", kind="tile", q=27, storage="f32", nx=384, ny=24, nz=128, steps=100, kinevisc=1e-3),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("flow",) * 7 + ("ensemble", "adjoint", "tile"))
    if kind == "flow":
        model, bnd = rng.choice((("reg", (1, 0, 12)), ("reg", (1, 0, 12)), ("reg", (1, 0, 11)), ("reg", (1, 11, 11)),
                                 ("reg", (1, 22, 12)), ("bgk", (0, 0, 11)), ("reg", (0, 0, 11)), ("reg", (0, 0, 0)),
                                 ("reg", (22, 11, 12)), ("bgk", (11, 21, 22))))
        cells = _log(rng, 4e3, 6e6)
        ry, rz = rng.uniform(0.25, 1.0), rng.uniform(0.2, 1.0)
        nx = (cells / (ry * rz)) ** (1 / 3)
        dims = [max(5, round(nx * r)) for r in (1.0, ry, rz)]
        dims[0] = max(dims[0], 24)
        inflow = bnd[0] == 1
        return _flow(None, dims, int(min(100, max(20, 2e8 / math.prod(dims)))), q=rng.choice((19, 27)), model=model,
                     storage=rng.choice(("f32", "f32", "f16s", "bf16s", "f64")), ibnd=bnd[0], jbnd=bnd[1], kbnd=bnd[2],
                     kinevisc=1.0 / 30.0 if model == "bgk" else 1e-3, cylinder=inflow and rng.random() < 0.5,
                     turbulence=inflow and rng.random() < 0.7,
                     readout=rng.choice(("moments", "moments", "averages", "restart")))
    if kind == "ensemble":
        big = rng.random() < 0.5
        n = [rng.randint(64, 140), rng.randint(48, 96), rng.randint(40, 90)] if big else \
            [rng.randint(20, 48), rng.randint(12, 32), rng.randint(10, 30)]
        return dict(kind=kind, members=rng.randint(4, 12) if big else rng.randint(8, 64), ni=n[0], nj=n[1], nk=n[2],
                    steps=50 if big else 200, storage=rng.choice(("f32", "f32", "f16s", "f64")))
    if kind == "adjoint":
        return dict(kind=kind, nx=rng.randint(64, 160), ny=rng.randint(24, 80), nz=rng.randint(24, 80),
                    steps=rng.choice((20, 40, 60)), every=rng.choice((5, 8, 10, 20)), storage=rng.choice(("f32", "f64")))
    return dict(kind=kind, q=rng.choice((19, 27)), storage=rng.choice(("f32", "f16s")), nx=rng.randint(100, 384),
                ny=rng.randint(10, 48), nz=rng.randint(40, 128), steps=50, kinevisc=1e-3)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _moments(dims, seed, u0):
    """rho, u, v, w on every cell, ghosts included: a mean flow and a few large-scale waves in every
    component, as an under-resolved turbulent state holds them."""
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    x, y, z = (torch.arange(n + 2, dtype=torch.float64, device=_device()) for n in (nx, ny, nz))
    out = []
    for mean, amp in ((1.0, 2e-3), (u0, 1.5e-2), (0.0, 1.5e-2), (0.0, 1.5e-2)):
        a = torch.full((nz + 2, ny + 2, nx + 2), mean, dtype=torch.float64, device=_device())
        for m in rng.integers(1, 4, (4, 3)):
            p = rng.uniform(0, 2 * np.pi, 3)
            a += 0.5 * amp * (torch.cos(2 * np.pi * m[2] * z / nz + p[2])[:, None, None]
                              * torch.cos(2 * np.pi * m[1] * y / ny + p[1])[None, :, None]
                              * torch.cos(2 * np.pi * m[0] * x / nx + p[0])[None, None, :])
        out.append(a)
    return out


def _slices(seed, ny, nz):
    """uu, vv, ww of the inflow turbulence, (NTURB + 1, nz, ny): smooth unit-variance slices that
    follow one another with correlation 0.98."""
    rng = np.random.default_rng(seed)
    noise = torch.from_numpy(rng.standard_normal((3, NTURB + 1, nz, ny))).to(_device())
    ky, kz = (2 * np.pi * torch.fft.fftfreq(n, dtype=torch.float64, device=_device()) for n in (ny, nz))
    s = torch.fft.ifft2(torch.fft.fft2(noise) * torch.exp(-16.0 * (kz[:, None] ** 2 + ky[None, :] ** 2))).real
    s = s - s.mean((2, 3), keepdim=True)
    s = s / (s.std((2, 3), keepdim=True) + 1e-30)
    for t in range(1, NTURB + 1):
        s[:, t] = 0.98 * s[:, t - 1] + math.sqrt(1 - 0.98 ** 2) * s[:, t]
    return s


def _box(dims, seed):
    """A solid block on the lower wall (ensemble members), inclusive 1-based bounds."""
    rng = np.random.default_rng(seed + 3)
    side = max(2, min(dims) // 6)
    lo = [int(dims[0] // 6 + rng.integers(0, max(1, dims[0] // 6))), int(rng.integers(1, dims[1] - side + 1)), 1]
    return [(l, l + side - 1) for l in lo]


def _mask(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    m = np.zeros((nz + 2, ny + 2, nx + 2), np.uint8)
    if c.get("cylinder"):
        # a cylinder along k, a quarter of the length downstream
        r = max(2, min(12, ny // 8))
        i, j = np.arange(nx + 2)[None, :], np.arange(ny + 2)[:, None]
        inside = (i - max(nx // 4, r + 2)) ** 2 + (j - ny // 2) ** 2 < r ** 2
        inside[:, [0, -1]] = False
        inside[[0, -1], :] = False
        m[:] = inside[None]
    elif c.get("block"):
        (i0, i1), (j0, j1), (k0, k1) = c["block"]
        m[k0:k1 + 1, j0:j1 + 1, i0:i1 + 1] = 1
    return m


def _turbines(c, seed):
    """Rotors in a row along i, the blade of the NREL 5-MW turbine, generic airfoil tables."""
    from lbm_amd import turbines
    rng = np.random.default_rng(seed + 5)
    deg = np.linspace(-180.0, 180.0, 73)
    foils = [np.stack([deg, a * np.sin(np.deg2rad(2 * deg)), 0.01 + 0.6 * np.sin(np.deg2rad(deg)) ** 2], 1)
             for a in (0.0, 0.05, 0.9, 0.95, 1.0, 1.05, 1.1, 1.15)]
    pos = [(c["nx"] * (1 + 2 * t) // (2 * c["turbines"] + 2), c["ny"] // 2, c["nz"] // 2, float(rng.uniform(-8, 8)), 3.0)
           for t in range(c["turbines"])]
    return turbines.from_infile(pos, 12.0, 0.0, TURBINE_LENGTH, TURBINE_VEL, foils, np.float32,
                                theta=rng.uniform(0, 2, c["turbines"]))


def _shear(nz):
    return ((np.arange(1, nz + 1) - 0.5) / nz) ** (1.0 / 7.0)


def _model(c):
    if c.get("model", "reg") == "bgk":
        return dict(ibgk=2)
    return dict(ibgk=3, ihrr=1, ivreman=1, smagorinsky=SMAGORINSKY)


def _member(c, seed, m):
    """Member m of an ensemble as a flow case: its sizes vary by up to a quarter."""
    rng = np.random.default_rng(1000 * c["ni"] + m)   # sizes belong to the case, not to the seed
    dims = [int(n * f) for n, f in zip((c["ni"], c["nj"], c["nk"]), rng.uniform(0.75, 1.0, 3))]
    f = _flow(None, dims, c["steps"], q=19, storage=c["storage"], kinevisc=1e-3, turbulence=True)
    return dict(f, block=_box(dims, seed + 17 * m)), seed + 17 * m


def _domain(c, seed):
    """A domain of a flow case with its inputs, started from the equilibrium of its moments."""
    dims = (c["nx"], c["ny"], c["nz"])
    d = Domain(c["q"], dims, c["storage"], kinevisc=c["kinevisc"], ibnd=c["ibnd"], jbnd=c["jbnd"], kbnd=c["kbnd"],
               iturb_pos=ITURB, **_model(c))
    inflow = c["ibnd"] == 1
    if inflow:
        d.set_inflow(UINI, 0.0, _shear(c["nz"]))
    if c["cylinder"] or c.get("block"):
        d.set_blanking(_mask(c, seed))
    if c["turbulence"] and not c["turbines"]:
        t = _slices(seed, c["ny"], c["nz"]).to(torch.float64 if c["storage"] == "f64" else torch.float32).cpu().numpy()
        d.set_turbulence(t[0], t[1], t[2], NTURB, AMPL)
    if c["turbines"]:
        d.set_turbines(_turbines(c, seed))
    d.init_equilibrium(*(a.cpu().numpy() for a in _moments(dims, seed, UINI if inflow else 0.02)))
    return d


def _tile_start(c, seed):
    """Equilibrium populations of a tile (periodic with itself along j), as a restart record holds them."""
    rho, u, v, w = _moments((c["nx"], c["ny"], c["nz"]), seed, UINI)
    e = _Lattice(c["q"]).equilibrium(rho, torch.stack((u, v, w)), True)
    e[:, :, 0], e[:, :, -1] = e[:, :, -2].clone(), e[:, :, 1].clone()
    return e


def prepare(case, seed):
    c = case
    if c["kind"] == "flow":
        d = _domain(c, seed)
        s = dict(case=c, dom=d, it=0, seed=seed)
        if c["readout"] == "restart":
            s["record"] = d.get_state()
        return s
    if c["kind"] == "ensemble":
        doms = [_domain(*_member(c, seed, m)) for m in range(c["members"])]
        return dict(case=c, doms=doms, ens=Ensemble(doms), it=0)
    if c["kind"] == "tile":
        d = Domain(c["q"], (c["nx"], c["ny"], c["nz"]), c["storage"], kinevisc=c["kinevisc"], ibnd=1, jbnd=BND_HALO,
                   kbnd=12, iturb_pos=ITURB, **_model(c))
        d.set_state(_tile_start(c, seed).permute(1, 2, 3, 0).to(torch.float32).cpu().numpy())
        d.set_inflow(UINI, 0.0, _shear(c["nz"]))
        nb = d.halo_bytes()
        snd, rcv = (torch.zeros(2 * nb, dtype=torch.uint8, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        return dict(case=c, dom=d, it=0, nb=nb, snd=snd, rcv=rcv, ext=torch.cuda.ExternalStream(d.stream_ptr()),
                    side=torch.cuda.Stream(), packed=torch.cuda.Event(), moved=torch.cuda.Event())
    p = _problem(c, seed)
    return dict(case=c, problem=p, force=p.force_field(p.a0), shear=p.shear_profile(p.c0))


def _problem(c, seed):
    nx = c["nx"]
    return ForcingProblem((nx, c["ny"], c["nz"]), c["storage"], c["steps"], c["every"], box_i=(nx // 3, nx - 12),
                          nblobs=16, i_blobs=nx // 4, seed=seed % 100000)


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(state):
    return {"flow": _run_flow, "ensemble": _run_ensemble, "tile": _run_tile, "adjoint": _run_adjoint}[state["case"]["kind"]](state)


def _run_flow(s):
    c, d, n = s["case"], s["dom"], s["case"]["steps"]
    if c["readout"] == "restart":
        d.set_state(s["record"])
        d.step(0, n)
        return d.get_state()
    it, s["it"] = s["it"], s["it"] + n
    if c["turbines"] and c["turbulence"]:
        d.generate_turbulence(NTURB, AMPL, s["seed"] + it, return_fields=False)
    if c["readout"] == "averages":
        d.set_averaging(True)
        d.step(it, n)
        return d.averages()[:4]
    d.step(it, n)
    return d.macrovars()


def _run_ensemble(s):
    it, s["it"] = s["it"], s["it"] + s["case"]["steps"]
    s["ens"].step(it, s["case"]["steps"])
    return _by_member([d.macrovars() for d in s["doms"]], np.concatenate)


def _by_member(moments, join):
    """rho, u, v, w of each member, or of all members end to end where that would be over 64 arrays."""
    if len(moments) <= 16:
        return moments
    return [join([a.reshape(-1) for a in f]) for f in zip(*moments)]


def _run_tile(s):
    d, nb, n = s["dom"], s["nb"], s["case"]["steps"]
    for it in range(s["it"] + 1, s["it"] + n + 1):
        d.step_part(it, PART_EDGE)
        d.halo_pack(2, s["snd"].data_ptr())
        s["packed"].record(s["ext"])
        d.step_part(it, PART_INNER)
        s["side"].wait_event(s["packed"])
        with torch.cuda.stream(s["side"]):   # where ranks send and receive; this tile is its own neighbour
            s["rcv"][:nb].copy_(s["snd"][nb:])
            s["rcv"][nb:].copy_(s["snd"][:nb])
            s["moved"].record(s["side"])
        s["ext"].wait_event(s["moved"])
        d.halo_unpack(2, s["rcv"].data_ptr())
    s["it"] += n
    # the tile's own planes of j: its ghost planes are the neighbours' cells
    return [a[:, 1:-1] for a in d.macrovars()]


def _run_adjoint(s):
    force, shear = s["force"].requires_grad_(True), s["shear"].requires_grad_(True)
    force.grad = shear.grad = None
    j = LatticeKE.apply(force, shear, s["problem"])
    j.backward()
    return j.detach(), force.grad, shear.grad


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    """Every step reads and writes each population once (an adjoint step reads the state and its
    adjoint and writes the adjoint); the averages read and write six sums a step; the readout
    is written once."""
    c = case
    size = {"f32": 4, "f64": 8, "f16s": 2, "bf16s": 2}[c["storage"]]
    real = 8 if c["storage"] == "f64" else 4
    q = c.get("q", 19)
    if c["kind"] == "ensemble":
        cells = sum(math.prod(_member(c, 0, m)[0][n] for n in ("nx", "ny", "nz")) for m in range(c["members"]))
    else:
        cells = c["nx"] * c["ny"] * c["nz"]
    per_step, flops, out = 2 * q * size, 20 * q, 4 * real
    if c["kind"] == "adjoint":
        per_step, flops, out = 5 * q * size + 48, 70 * q, 48
    elif c.get("readout") == "averages":
        per_step += 12 * real
    elif c.get("readout") == "restart":
        out = 2 * q * real
    return dict(bytes=cells * (c["steps"] * per_step + out), flops=cells * c["steps"] * flops)


# ---------------------------------------------------------------------------------------------
# the same in 64 bits: the lattice update on whole arrays with all its ghost layers
# ---------------------------------------------------------------------------------------------
CX = (0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, -1, 1, 0, 0, -1, 1, 0, 0, -1, 1, -1, 1, 1, -1, -1, 1)
CY = (0, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 1, -1, 0, 0, -1, 1, 1, -1, -1, 1, 1, -1, 1, -1)
CZ = (0, 0, 0, 0, 0, -1, 1, 0, 0, 0, 0, -1, 1, 1, -1, 1, -1, 1, -1, 1, -1, -1, 1, -1, 1, -1, 1)
IN = slice(1, -1)
PAIRS = ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))


class _Lattice:
    def __init__(self, q):
        self.q = q
        self.c = list(zip(CX, CY, CZ))[:q]
        den = {19: (1 / 3, 1 / 18, 1 / 36), 27: (8 / 27, 2 / 27, 1 / 54, 1 / 216)}[q]
        self.w = [den[sum(abs(x) for x in c)] for c in self.c]
        self.find = {c: l for l, c in enumerate(self.c)}
        self.opp = [self.find[(-x, -y, -z)] for x, y, z in self.c]
        self.C = torch.tensor(self.c, dtype=torch.float64, device=_device())
        self.W = torch.tensor(self.w, dtype=torch.float64, device=_device())[:, None]
        # c c in the order xx, yy, zz, xy, xz, yz
        self.CC = torch.stack([self.C[:, p] * self.C[:, r] for p, r in PAIRS], 1)
        self.one = torch.ones(1, q, dtype=torch.float64, device=_device())

    @staticmethod
    def mm(m, f):
        """A small matrix times fields stacked along the first axis."""
        return torch.mm(m, f.reshape(f.shape[0], -1)).reshape((m.shape[0],) + f.shape[1:])

    def equilibrium(self, rho, vel, third):
        usq = (vel * vel).sum(0)
        cu = self.mm(self.C, vel)
        p = 1.0 - 1.5 * usq + cu * (3.0 + 4.5 * cu)
        if third:
            p[1:] += 4.5 * cu[1:] * (cu[1:] * cu[1:] - usq)
        shape = (self.q,) + (1,) * (p.dim() - 1)
        return self.W.reshape(shape) * rho * p

    def moments(self, f):
        """rho and the velocity, (4, ...)."""
        m = self.mm(torch.cat((self.one, self.C.t())), f)
        return torch.cat((m[:1], m[1:] / m[:1]))


class _Steps:
    """The update of one flow case: f1 holds the state, f2 the state before it, both (q, nz+2, ny+2, nx+2)."""

    def __init__(self, c, force=None, shear=None):
        self.c, self.lat = c, _Lattice(c["q"])
        self.n = (c["nx"], c["ny"], c["nz"])
        self.third = c["model"] == "reg"
        nz = c["nz"]
        self.shear = torch.from_numpy(_shear(nz)).to(_device()) if shear is None else shear
        self.solid = None
        self.turb = None
        self.force = force
        self.rotors = None

    # -- boundaries --------------------------------------------------------------------------
    def _plane(self, axis, at, rest=IN, shift=(0, 0, 0)):
        """Index (k, j, i) of a plane of an axis, its tangential cells shifted by -shift."""
        idx = []
        for d in (2, 1, 0):
            if d == axis:
                idx.append(at)
            elif rest is IN:
                lo = 1 - shift[d]
                idx.append(slice(lo, lo + self.n[d]))
            else:
                idx.append(rest)
        return tuple(idx)

    def _periodic(self, f):
        for d, code in enumerate((self.c["ibnd"], self.c["jbnd"], self.c["kbnd"])):
            if code == 0:
                for ghost, src in ((0, self.n[d]), (self.n[d] + 1, 1)):
                    f[(slice(None),) + self._plane(d, ghost, slice(None))] = \
                        f[(slice(None),) + self._plane(d, src, slice(None))].clone()

    def _closed(self, f1, f2, d, side, slip):
        ghost, wall = (self.n[d] + 1, self.n[d]) if side else (0, 1)
        g = self._plane(d, ghost)
        out = [(l, c) for l, c in enumerate(self.lat.c) if c[d] == (1 if side else -1)]
        new = []
        for l, c in out:
            m = self.lat.find[tuple(-x if a == d else slip * x for a, x in enumerate(c))]
            new.append((m, f2[(l,) + g].clone()))
        for l, c in out:
            new.append((l, f1[(l,) + self._plane(d, wall, IN, c)].clone()))
        for l, v in new:
            f1[(l,) + g] = v

    def _ghost_set(self, f1, f2, at, mirror):
        """An edge or a corner: at has None on the axis that it runs along."""
        sgn = [0 if a is None else (1 if a else -1) for a in at]
        pos = lambda c: tuple(IN if at[d] is None else (self.n[d] + 1 if at[d] else 0) - c[d] for d in (2, 1, 0))  # noqa: E731
        out = [(l, c) for l, c in enumerate(self.lat.c) if all(s == 0 or s * x > 0 for s, x in zip(sgn, c))]
        g = pos((0, 0, 0))
        for l, c in out:
            m = self.lat.find.get(tuple(s * x for s, x in zip(mirror, c)))
            if m is not None:
                f1[(m,) + g] = f2[(l,) + g]
        for l, c in out:
            f1[(l,) + g] = f1[(l,) + pos(c)]

    def _edges(self, f1, f2):
        b = (self.c["ibnd"], self.c["jbnd"], self.c["kbnd"])
        opt = lambda x, y: 1 if b[x] == 22 and b[y] == 22 else -1   # noqa: E731
        order = ((0, 0), (1, 0), (0, 1), (1, 1))
        if b[1] > 10 and b[2] > 10:
            for j, k in order:
                # the upper-upper edge keeps the velocity along it, as the reference's does
                self._ghost_set(f1, f2, (None, j, k), (1 if j and k else opt(1, 2), -1, -1))
        if b[0] > 10 and b[1] > 10:
            for i, j in order:
                self._ghost_set(f1, f2, (i, j, None), (-1, -1, opt(0, 1)))
        if b[0] > 10 and b[2] > 10:
            for i, k in order:
                self._ghost_set(f1, f2, (i, None, k), (-1, opt(0, 2), -1))
        if min(b) > 10:
            # the reference's list of corners, read column by column
            nx, ny, nz = (x + 1 for x in self.n)
            t = (0, 0, 0, 0, 0, nz, 0, ny, 0, 0, ny, nz, nx, 0, 0, nx, 0, nz, nx, ny, 0, nx, ny, nz)
            for m in range(8):
                at = (t[m], t[8 + m], t[16 + m])
                if all(a in (0, n + 1) for a, n in zip(at, self.n)):
                    self._ghost_set(f1, f2, tuple(int(a > 0) for a in at), (-1, -1, -1))

    def boundaries(self, f1, f2):
        self._periodic(f1)
        for d, code in enumerate((self.c["ibnd"], self.c["jbnd"], self.c["kbnd"])):
            if code > 10:
                self._closed(f1, f2, d, 0, 1 if code // 10 == 2 else -1)
                self._closed(f1, f2, d, 1, 1 if code % 10 == 2 else -1)
        self._edges(f1, f2)
        if self.c["ibnd"] == 1:
            inner = f1[:, IN, IN, 1].clone()
            speed = (UINI * self.shear)[:, None]
            for l, c in enumerate(self.lat.c):
                s = l if c[0] <= 0 else self.lat.opp[l]
                f1[l, IN, IN, 0] = inner[s] - 6.0 * self.lat.w[s] * self.lat.c[s][0] * speed
            f1[:, IN, IN, -1] = f1[:, IN, IN, -2].clone()
        self._periodic(f1)

    # -- interior ------------------------------------------------------------------------------
    def collide(self, f, mom, it):
        """Post-collision populations of the interior cells from their populations and moments."""
        c, lat = self.c, self.lat
        rho, vel = mom[0], mom[1:]
        feq = lat.equilibrium(rho, vel, self.third)
        if c["model"] == "bgk":
            tau = 3.0 * c["kinevisc"] + 0.5
            out = feq + (1.0 - 1.0 / tau) * (f - feq)
        else:
            ne = f - feq
            a = lat.mm(lat.CC.t(), ne)
            trace = ne.sum(0) / 3.0
            xx, yy, zz, xy, xz, yz = a[0] - trace, a[1] - trace, a[2] - trace, a[3], a[4], a[5]
            mag = (xx * xx + yy * yy + zz * zz + 2.0 * (xy * xy + xz * xz + yz * yz)).clamp_min(2.3e-308)
            b11, b22, b33 = xx * xx + xy * xy + xz * xz, xy * xy + yy * yy + yz * yz, xz * xz + yz * yz + zz * zz
            b12, b13, b23 = xx * xy + xy * yy + xz * yz, xx * xz + xy * yz + xz * zz, xy * xz + yy * yz + yz * zz
            t = (b11 * b22 - b12 * b12 + b11 * b33 - b13 * b13 + b22 * b33 - b23 * b23) / mag
            some = t > 1.5e-154
            eddy = torch.where(some, 2.5 * SMAGORINSKY ** 2 * torch.sqrt(torch.where(some, t, torch.ones_like(t))),
                               torch.zeros_like(t))
            fac = 1.0 - 1.0 / (3.0 * (c["kinevisc"] + eddy) + 0.5)
            tr = xx + yy + zz
            g = torch.stack((xx * vel[0] + xy * vel[1] + xz * vel[2], xy * vel[0] + yy * vel[1] + yz * vel[2],
                             xz * vel[0] + yz * vel[1] + zz * vel[2]))
            cac = lat.mm(lat.CC, torch.stack((xx, yy, zz, 2.0 * xy, 2.0 * xz, 2.0 * yz)))
            n = cac - tr / 3.0 + lat.mm(lat.C, vel) * (3.0 * cac - tr) - 2.0 * lat.mm(lat.C, g)
            out = feq + fac * (4.5 * lat.W[:, :, None, None]) * n
        if self.turb is not None:
            s = it % NTURB or NTURB
            m = mom[:, :, :, ITURB - 1]
            out[:, :, :, ITURB - 1] += lat.equilibrium(m[0], m[1:] + AMPL * self.turb[:, s], self.third) - \
                lat.equilibrium(m[0], m[1:], self.third)
        force = self.force if self.rotors is None else self.rotors.force(mom)
        if force is not None:
            out = out + lat.equilibrium(rho, vel - force.movedim(-1, 0) / rho, False) - lat.equilibrium(rho, vel, False)
        if self.solid is not None:
            out = torch.where(self.solid, out[self.lat.opp], out)
        return out

    def step(self, f1, f2, it, mom=None):
        """(f1, f2) after step it; mom: moments to collide with instead of the populations' own."""
        inner = (slice(None), IN, IN, IN)
        x = f1[inner]
        mom = self.lat.moments(x) if mom is None else mom
        f1 = f1.clone()
        f1[inner] = self.collide(x, mom, it)
        f2 = f2.clone()
        self.boundaries(f1, f2)
        new = []
        for l, (cx, cy, cz) in enumerate(self.lat.c):
            nx, ny, nz = self.n
            new.append(f1[l, 1 - cz:1 - cz + nz, 1 - cy:1 - cy + ny, 1 - cx:1 - cx + nx])
        f2[inner] = torch.stack(new)
        return f2, f1


class _Rotors:
    """Actuator lines: forces of the blade sections at their points and their Gaussian deposit."""

    def __init__(self, t, n):
        self.t, self.n = t, n
        self.theta = np.array(t["theta"], np.float64)
        self.krad = min(5, math.ceil(3.0 * math.sqrt(2.0)))

    def force(self, mom):
        t = self.t
        self.theta = self.theta + np.asarray(t["omegand"], np.float64)
        nx, ny, nz = self.n
        F = torch.zeros((nz, ny, nx, 3), dtype=torch.float64, device=_device())
        relm, chord, dc, twist = (np.asarray(t[k], np.float64) for k in ("relm", "chord", "dc", "twist"))
        pos, frame = [], []
        for r in range(len(self.theta)):
            yaw, tilt = float(t["yaw"][r]), float(t["tilt"][r])
            ea = np.array([math.cos(yaw) * math.cos(tilt), math.sin(yaw) * math.cos(tilt), -math.sin(tilt)])
            e1 = np.array([-math.sin(yaw), math.cos(yaw), 0.0])
            e2 = np.array([-math.cos(yaw) * math.sin(tilt), -math.sin(yaw) * math.sin(tilt), -math.cos(tilt)])
            for b in range(t["nblades"]):
                th = self.theta[r] + 2 * math.pi * b / t["nblades"]
                for s in range(len(relm)):
                    pos.append(np.asarray(t["hub"][r], np.float64) + relm[s] * (math.cos(th) * e1 + math.sin(th) * e2))
                    frame.append((r, th, ea, -math.sin(th) * e1 + math.cos(th) * e2, s))
        pos = np.array(pos)
        cell = np.floor(pos).astype(int)
        fr = torch.from_numpy(pos - cell).to(_device())
        base = torch.from_numpy(np.clip(cell, 1, np.array(self.n) - 1) - 1).to(_device())
        vals = []
        for field in mom:
            v = 0.0
            for corner in range(8):
                o = [(corner >> d) & 1 for d in range(3)]
                wgt = math.prod([fr[:, d] if o[d] else 1.0 - fr[:, d] for d in range(3)], start=1.0)
                v = v + wgt * field[base[:, 2] + o[2], base[:, 1] + o[1], base[:, 0] + o[0]]
            vals.append(v)
        vals = torch.stack(vals).cpu().numpy()
        for p, (r, th, ea, et, s) in enumerate(frame):
            dens, ux, uy, uz = vals[:, p]
            ut = float(t["omegand"][r]) * relm[s] - uz * math.cos(th) - uy * math.sin(th)
            phi = math.atan2(ux, ut)
            ang = math.degrees(phi) - twist[s] - float(t["pitch"][r])
            tab = np.asarray(t["foils"][t["nfoil"][s] - 1], np.float64)
            inside = tab[0, 0] < ang <= tab[-1, 0]
            cl, cd = (np.interp(ang, tab[:, 0], tab[:, k]) if inside else 0.0 for k in (1, 2))
            q = 0.5 * dens * (ux * ux + ut * ut) * chord[s] * dc[s]
            fp = q * cl * (math.cos(phi) * ea + math.sin(phi) * et) - q * cd * (math.sin(phi) * ea - math.cos(phi) * et)
            rng = [(max(1, int(cell[p, d]) - self.krad), min(self.n[d], int(cell[p, d]) + self.krad)) for d in range(3)]
            if any(lo > hi for lo, hi in rng):
                continue
            e = [torch.exp(-(torch.arange(lo, hi + 1, dtype=torch.float64, device=_device()) - pos[p, d]) ** 2 / 4.0)
                 for d, (lo, hi) in enumerate(rng)]
            wgt = e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
            sl = tuple(slice(lo - 1, hi) for lo, hi in reversed(rng))
            F[sl] += (wgt / wgt.sum())[..., None] * torch.from_numpy(fp).to(_device())
        return F


def _phases(seed, n):
    """2 pi U of the SplitMix64 stream."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return 2 * np.pi * (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _generated(seed, ny, nz):
    """The inflow turbulence that the generator draws: a Gaussian spectrum with random phases, transformed and
    chained in time, (3, NTURB + 1, nz, ny)."""
    n1, n2, ns = ny + ny % 2, nz + nz % 2, NTURB + 1
    nh = n1 // 2 + 1
    r2 = 8.0 / (10.0 / math.sqrt(3.0)) ** 2
    kap, lam = (2.0 * 3.141592653589 / n for n in (n1, n2))
    l, p = np.arange(nh), np.where(np.arange(n2) < n2 // 2, np.arange(n2), np.arange(n2) - n2)
    dk = (2.0 * 3.141592653589) ** 2 / (n1 * n2)
    lf, pf = np.arange(-n1 // 2 + 1, n1 // 2 + 1), np.arange(-n2 // 2 + 1, n2 // 2 + 1)
    total = np.exp(-2.0 * (kap ** 2 * lf[None, :] ** 2 + lam ** 2 * pf[:, None] ** 2) / r2).sum() - 1.0
    amp = np.sqrt(dk) * np.sqrt(1.0 / (dk * total)) * np.exp(-(kap ** 2 * l[None, :] ** 2 + lam ** 2 * p[:, None] ** 2) / r2)
    amp[0, 0] = 0.0
    phi = _phases(seed, 3 * ns * nh * n2).reshape(3 * ns, nh, n2).transpose(0, 2, 1)
    x = torch.from_numpy(amp * np.exp(1j * phi)).to(_device()).reshape(3, ns, n2, nh)
    z = torch.fft.ifft(x, dim=2, norm="forward")
    y = torch.fft.irfft(z, n=n1, dim=3, norm="forward")[:, :, :nz, :ny].contiguous()
    for t in range(1, ns):
        s = 0.98 * y[:, t - 1] + math.sqrt(1 - 0.98 ** 2) * y[:, t]
        s = s - s.mean((1, 2), keepdim=True)
        y[:, t] = s / torch.sqrt((s * s).sum((1, 2), keepdim=True) / (ny * nz - 1))
    return y


def _start(c, seed):
    """A flow case before its first step: the update, both buffers and the moments it started from."""
    st = _Steps(c)
    if c["cylinder"] or c.get("block"):
        st.solid = torch.from_numpy(_mask(c, seed)[1:-1, 1:-1, 1:-1].astype(bool)).to(_device())
    if c["turbines"]:
        st.rotors = _Rotors(_turbines(c, seed), st.n)
    if c["turbulence"]:
        st.turb = _generated(seed, c["ny"], c["nz"]) if c["turbines"] else _slices(seed, c["ny"], c["nz"])
    mom = _moments(st.n, seed, UINI if c["ibnd"] == 1 else 0.02)
    clamp = [torch.arange(n + 2, device=_device()).clamp(1, n) for n in reversed(st.n)]
    mom = torch.stack([m[clamp[0]][:, clamp[1]][:, :, clamp[2]] for m in mom])
    f2 = st.lat.equilibrium(mom[0], mom[1:], st.third)
    f1 = f2.clone()
    st.boundaries(f2, f1)
    st.boundaries(f1, f2)
    return st, f1, f2, mom[:, IN, IN, IN]


def _exact_flow(c, seed):
    st, f1, f2, mom = _start(c, seed)
    if c["readout"] == "restart":
        # the record holds the equilibrium start; what is read back is collided with its own moments
        f2, mom = f1.clone(), None
    sums = 0.0
    for it in range(1, c["steps"] + 1):
        f1, f2 = st.step(f1, f2, it, mom)
        mom = None
        if c["readout"] == "averages":
            v = st.lat.moments(f1[:, IN, IN, IN])[1:]
            sums = sums + torch.cat((v, v * v))
    if c["readout"] == "restart":
        return f1.permute(1, 2, 3, 0).contiguous()
    if c["readout"] == "averages":
        m = torch.zeros((4,) + f1.shape[1:], dtype=torch.float64, device=_device())
        mean = sums / c["steps"]
        m[:3, IN, IN, IN] = mean[:3]
        m[3, IN, IN, IN] = torch.sqrt((mean[3:] - mean[:3] ** 2).clamp_min(0).sum(0) / 3.0)
        return list(m)
    return list(st.lat.moments(f1))


def _exact_tile(c, seed):
    f = dict(FLOW, **{k: c[k] for k in ("q", "storage", "nx", "ny", "nz", "steps", "kinevisc")})
    st = _Steps(f)
    f1 = _tile_start(c, seed).to(torch.float32).to(torch.float64)
    f2 = f1.clone()
    for it in range(1, c["steps"] + 1):
        f1, f2 = st.step(f1, f2, it)
    return [m[:, IN] for m in st.lat.moments(f1)]


def _exact_adjoint(c, seed):
    p = dict(FLOW, q=19, storage=c["storage"], nx=c["nx"], ny=c["ny"], nz=c["nz"], steps=c["steps"])
    problem = _problem(c, seed)
    f1 = torch.from_numpy(np.ascontiguousarray(problem.f0.transpose(3, 0, 1, 2))).to(torch.float64).to(_device())
    (i0, i1), box = problem.box[0], (slice(None), IN, IN)
    F, s = problem.force_field(problem.a0), problem.shear_profile(problem.c0)
    problem.close()
    force = F.to(_device()).requires_grad_(True)
    shear = s.to(_device()).requires_grad_(True)
    with torch.no_grad():
        f1, f2 = _Steps(p, shear=shear.detach()).step(f1, f1.clone(), 1)

    def advance(a, b, force, shear):
        a, b = _Steps(p, force[IN, IN, IN], shear).step(a, b, 0)
        rho, u, v, w = _Lattice(19).moments(a[box + (slice(i0, i1 + 1),)])
        return a, b, (0.5 * rho * (u * u + v * v + w * w)).mean()

    total = 0.0
    for _ in range(c["steps"]):
        f1, f2, e = checkpoint(advance, f1, f2, force, shear, use_reentrant=False)
        total = total + e / c["steps"]
    total.backward()
    grad = torch.zeros_like(force)
    grad[IN, IN, IN] = force.grad[IN, IN, IN]
    return total.detach(), grad, shear.grad


def exact(case, seed):
    c = case
    if c["kind"] == "ensemble":
        if c["members"] * c["steps"] > 6000:
            return None   # a minute of small launches
        return _by_member([_exact_flow(*_member(c, seed, n)) for n in range(c["members"])], torch.cat)
    return {"flow": _exact_flow, "tile": _exact_tile, "adjoint": _exact_adjoint}[c["kind"]](c, seed)
