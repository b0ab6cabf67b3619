"""What a program that uses this framework has it do, as cases that can be
timed and whose results can be compared.

Kinds, each through the public entry points of vpic_amd:

  step      Simulation.advance() over one sort interval (a sort, then the
            interval's steps): periodic plasma, or a 2D current sheet
            between conducting, reflecting walls
  push      the particle half of a sort interval in given fields
  vacuum    Simulation.advance() of a run without particles
  diag      the energies and the charge-conservation error of a time step
  hydro     the moment dump of both species
  collide   binary collisions of both species (sorted first, as they need)
  ensemble  a batch of small boxes stepped together
  adjoint   the magnetic energy after n steps and its gradients, FP32/FP64

Particles come from torch's generator and `seed` alone; exact() repeats the
method in plain torch in 64 bits.
"""
import math

import numpy as np
import torch

DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # a box of a unit-test deck: latency and launches are all of it
        dict(name="step_smallest", kind="step", nx=12, ny=10, nz=9, ppc=8,
             steps=10, walls=False),
        # the cubic validation box, two species of 64 per cell
        dict(name="step_box32", kind="step", nx=32, ny=32, nz=32, ppc=64,
             steps=20, walls=False),
        # a reconnection sheet: 2D, walls, density far from uniform
        dict(name="step_sheet", kind="step", nx=512, ny=1, nz=257, ppc=48,
             steps=20, walls=True),
        # production plasma, as the repository's benchmark sizes it
        dict(name="step_plasma", kind="step", nx=256, ny=128, nz=128, ppc=100,
             steps=20, walls=False),
        # tracers in given fields on an odd box
        dict(name="push_odd", kind="push", nx=97, ny=61, nz=83, ppc=40,
             steps=10),
        # an electromagnetic run before any plasma is loaded
        dict(name="vacuum", kind="vacuum", nx=257, ny=150, nz=128, steps=20),
        # energies and div E error of one dump step
        dict(name="diag", kind="diag", nx=64, ny=64, nz=64, ppc=64),
        # hydro dump of electrons and ions
        dict(name="hydro", kind="hydro", nx=72, ny=64, nz=50, ppc=64),
        # electron-ion and electron-electron collisions of one step
        dict(name="collide", kind="collide", nx=48, ny=48, nz=48, ppc=64),
        # a parameter scan of small 2D beam boxes
        dict(name="ensemble", kind="ensemble", boxes=48, side=64, ppc=64,
             steps=20),
        # gradient of a Weibel run's magnetic energy
        dict(name="adjoint_f32", kind="adjoint", nx=64, ny=64, nz=64, ppc=32,
             steps=20, ckpt=10, bits=32),
        # the same in double, on a small odd box
        dict(name="adjoint_f64", kind="adjoint", nx=21, ny=34, nz=17, ppc=16,
             steps=12, ckpt=5, bits=64),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(cells_lo, cells_hi, side_lo=6, side_hi=256):
        while True:
            n = [size(side_lo, side_hi) for _ in range(3)]
            if cells_lo <= n[0] * n[1] * n[2] <= cells_hi:
                return dict(nx=n[0], ny=n[1], nz=n[2])

    def ppc_for(cells, lo, hi, most):
        return max(lo, min(size(lo, hi), most // cells))

    kind = rng.choice(("step", "step", "sheet", "push", "vacuum", "diag",
                       "hydro", "collide", "ensemble", "adjoint"))
    if kind == "step":
        b = box(500, 2000000)
        cells = b["nx"] * b["ny"] * b["nz"]
        return dict(kind="step", ppc=ppc_for(cells, 4, 120, 100000000),
                    steps=rng.choice((10, 20, 25)), walls=False, **b)
    if kind == "sheet":
        nx, nz = size(48, 1024), size(24, 512)
        return dict(kind="step", nx=nx, ny=1, nz=nz,
                    ppc=ppc_for(nx * nz, 16, 200, 40000000),
                    steps=rng.choice((10, 20, 25)), walls=True)
    if kind == "push":
        b = box(1000, 2000000)
        cells = b["nx"] * b["ny"] * b["nz"]
        return dict(kind="push", ppc=ppc_for(cells, 4, 120, 40000000),
                    steps=rng.choice((5, 10, 20)), **b)
    if kind == "vacuum":
        return dict(kind="vacuum", steps=rng.choice((10, 20)),
                    **box(2000, 6000000))
    if kind in ("diag", "hydro", "collide"):
        b = box(500, 500000, 6, 128)
        cells = b["nx"] * b["ny"] * b["nz"]
        return dict(kind=kind, ppc=ppc_for(cells, 4, 128, 20000000), **b)
    if kind == "ensemble":
        return dict(kind="ensemble", boxes=size(4, 96), side=size(24, 96),
                    ppc=size(16, 128), steps=rng.choice((10, 20)))
    b = box(500, 150000, 6, 96)
    cells = b["nx"] * b["ny"] * b["nz"]
    return dict(kind="adjoint", ppc=ppc_for(cells, 4, 64, 4000000),
                steps=rng.choice((8, 12, 20)), ckpt=rng.choice((4, 5, 10)),
                bits=rng.choice((32, 32, 64)), **b)


# ---------------------------------------------------------------------------
# inputs (torch and the seed only)
# ---------------------------------------------------------------------------

class Geo:
    """Sizes and constants of a box of cells d_e wide (1/8 d_e for the sheet,
    1/2 for the beams, 1/10 for the Weibel box), dt just under Courant,
    natural units (c = eps0 = m_e = |q_e| = n0 = 1)."""

    def __init__(self, nx, ny, nz, d, walls=False):
        self.n = (nx, ny, nz)
        self.d = d
        self.walls = walls
        self.l = tuple(d * k for k in self.n)
        dims = sum(1 for k in self.n if k > 1)
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        self.dt = f32(0.95 * d / math.sqrt(max(dims, 1)))
        self.rd = f32(1.0 / d)
        self.dV = f32(d ** 3)
        self.r8V = f32(0.125 / d ** 3)
        self.nv = (nx + 2) * (ny + 2) * (nz + 2)
        self.cells = nx * ny * nz

    def grid(self):
        from vpic_amd import types as T
        (lx, ly, lz), (nx, ny, nz) = self.l, self.n
        g = T.grid_periodic(0, 0, 0, lx, ly, lz, nx, ny, nz, self.dt)
        if self.walls:
            for k in (0, 3):
                g.fbc[k] = T.BC_PEC_FIELDS
                g.pbc[k] = T.BC_REFLECT_PARTICLES
        return g

    def voxel(self, x, y, z):
        return x + (self.n[0] + 2) * (y + (self.n[1] + 2) * z)


def geo(case):
    k = case["kind"]
    if k == "adjoint":
        return Geo(case["nx"], case["ny"], case["nz"], 0.1)
    if case.get("walls"):
        return Geo(case["nx"], 1, case["nz"], 0.125, True)
    return Geo(case["nx"], case["ny"], case["nz"], 1.0)


def generator(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(((int(seed) * 1000003 + stream) * 2654435761) % (1 << 62))
    return g


CHUNK = 1 << 24  # particles generated at a time


def cell_voxels(G, first, count, ppc):
    c = torch.arange(first, first + count, device=DEV) // ppc
    nx, ny, _ = G.n
    return G.voxel(1 + c % nx, 1 + (c // nx) % ny, 1 + c // (nx * ny))


def fill_thermal(out, G, ppc, uth, seed, stream, drift=None, w=None,
                 half=None):
    """Rows of `out` (n, 8 words of particle_t, float32): ppc per cell, cell
    by cell, uniform in the cell, momenta N(drift, uth) per axis; with `half`
    the second half of every cell drifts the other way."""
    r = generator(seed, stream)
    n = out.shape[0]
    w = 1.0 / ppc if w is None else w
    for a in range(0, n, CHUNK):
        o = out[a:a + CHUNK]
        m = o.shape[0]
        o[:, 0:3] = torch.rand((m, 3), generator=r, device=DEV) * 2 - 1
        o.view(torch.int32)[:, 3] = cell_voxels(G, a, m, ppc).to(torch.int32)
        u = torch.randn((m, 3), generator=r, device=DEV)
        u *= torch.tensor(uth, device=DEV)
        if drift is not None:
            u[:, 0] += drift
            if half:
                k = torch.arange(a, a + m, device=DEV) % ppc
                u[:, 0] -= 2 * drift * (k >= ppc // 2)
        o[:, 4:7] = u
        o[:, 7] = w


def fill_sheet(out, G, q, m, uth, ud, seed, stream):
    """A current sheet (density sech^2 of half-thickness lx / 25) on a
    background of a fifth of its peak, drifting along y, in load order."""
    r, xr = generator(seed, stream), generator(seed, 900)  # pairs share x
    nx, _, nz = G.n
    lx = nx * G.d
    L = lx / 25
    n = out.shape[0]
    sheet = 2 * L * math.tanh(0.5 * lx / L)
    ns = int(n * sheet / (sheet + 0.2 * lx))
    w = (sheet + 0.2 * lx) * G.d * (nz * G.d) / n
    for a in range(0, n, CHUNK):
        o = out[a:a + CHUNK]
        k = o.shape[0]
        s = torch.arange(a, a + k, device=DEV) < ns
        v = torch.rand((k, 3), generator=xr, device=DEV, dtype=torch.float64)
        t = math.tanh(0.5 * lx / L)
        x = torch.where(s, L * torch.atanh((2 * v[:, 0] - 1) * t) + 0.5 * lx,
                        v[:, 0] * lx) / G.d
        z = v[:, 2] * nz
        cx = x.floor().clamp(0, nx - 1)
        cz = z.floor().clamp(0, nz - 1)
        o[:, 0] = (2 * (x - cx) - 1).clamp(-1, 1).float()
        o[:, 1] = (2 * v[:, 1] - 1).float()
        o[:, 2] = (2 * (z - cz) - 1).clamp(-1, 1).float()
        o.view(torch.int32)[:, 3] = G.voxel(1 + cx.int(), 1, 1 + cz.int())
        u = uth * torch.randn((k, 3), generator=r, device=DEV)
        u[:, 1] += ud * s
        o[:, 4:7] = u
        o[:, 7] = w


def fill_fields(f, G, amplitude, seed, electric=1.0):
    """E and cB of every record (n, 20 words of field_t): smooth waves of a
    few periods along each axis, of random phase, plus 1% noise; E weaker
    than cB by `electric`."""
    r = generator(seed, 77)
    nx, ny, nz = G.n
    f.zero_()
    v = f.view(nz + 2, ny + 2, nx + 2, 20)
    ax = [2 * math.pi * torch.arange(k + 2, device=DEV) / k for k in G.n]
    ph = torch.rand((6, 3), generator=r, device=DEV) * 2 * math.pi
    wrap = [(torch.arange(k + 2, device=DEV) - 1) % k for k in G.n]
    for c in range(6):
        wave = (torch.sin(ax[0] + ph[c, 0])[None, None, :] +
                torch.sin(2 * ax[1] + ph[c, 1])[None, :, None] +
                torch.sin(ax[2] + ph[c, 2])[:, None, None])
        noise = torch.randn((nz, ny, nx), generator=r, device=DEV)
        noise = noise[wrap[2]][:, wrap[1]][:, :, wrap[0]]
        v[..., c if c < 3 else c + 1] = amplitude * (
            electric if c < 3 else 1.0) * (wave + 0.01 * noise)


# E against cB of the push cases: their fields stand still, and a stronger E
# would heat the tracers without bound from pass to pass
TRACER_E = 0.02


def drift_of(p, G, uth, seed, stream):
    """Positions some steps after a sort: every particle moved along each
    axis by a normal displacement of 8 steps at uth, across periodic faces
    (a copy of p)."""
    r = generator(seed, stream)
    out = p.clone()
    for a in range(0, out.shape[0], CHUNK):
        o = out[a:a + CHUNK]
        s = 8 * uth * G.dt * G.rd
        i = o.view(torch.int32)[:, 3].long()
        c = [None] * 3
        c[0] = i % (G.n[0] + 2)
        c[1] = (i // (G.n[0] + 2)) % (G.n[1] + 2)
        c[2] = i // ((G.n[0] + 2) * (G.n[1] + 2))
        for k in range(3):
            x = (o[:, k].double() + 1) / 2 + s * torch.randn(
                o.shape[0], generator=r, device=DEV, dtype=torch.float64)
            m = x.floor()
            o[:, k] = (2 * (x - m) - 1).float().clamp(-1, 1)
            c[k] = (c[k] - 1 + m.long()) % G.n[k] + 1
        o.view(torch.int32)[:, 3] = G.voxel(*c).int()
    return out


def words(n, w):
    return torch.empty((n, w), dtype=torch.float32, device=DEV)


# (name, charge, mass, thermal momentum, drift) of the two species
ELECTRON = ("electron", -1.0, 1.0, 0.1)
ION = ("ion", 1.0, 25.0, 0.02)


def fill_species(case, G, seed, k, out):
    name, q, m, uth = (ELECTRON, ION)[k]
    if case.get("walls"):
        # Ti/Te = 5, wpe/wce = 3
        uth, ud = ((0.0962, 0.0222), (0.0430, -0.111))[k]
        fill_sheet(out, G, q, m, uth, ud, seed, 10 + k)
    else:
        fill_thermal(out, G, case["ppc"], (uth,) * 3, seed, 10 + k)


def sheet_fields(f, G, seed):
    """B_z of the sheet with a perturbation of random phase."""
    r = generator(seed, 78)
    nx, _, nz = G.n
    f.zero_()
    v = f.view(nz + 2, 3, nx + 2, 20)
    lx = nx * G.d
    x = (torch.arange(nx + 2, device=DEV) - 0.5) * G.d - 0.5 * lx
    z = 2 * math.pi * torch.arange(nz + 2, device=DEV) / nz
    ph = torch.rand(1, generator=r, device=DEV) * 2 * math.pi
    v[:, 1, :, 6] = torch.tanh(x * 25 / lx)[None, :] / 3
    v[:, 1, :, 4] = 0.03 * (torch.sin(z + ph)[:, None] *
                            torch.cos(math.pi * x / lx)[None, :])


def beam_boxes(case):
    """(nx, ny, ppc, drift) of every box of the batch: sides, counts and
    drifts differ from box to box around the case's."""
    out = []
    for b in range(case["boxes"]):
        s, p = case["side"], case["ppc"]
        out.append((max(8, s + 16 * ((b * 5) % 7 - 3)),
                    max(8, s + 16 * ((b * 3) % 5 - 2)),
                    max(4, p // 2 + (b * 37) % p),
                    0.05 + 0.25 * ((b * 11) % 17) / 16))
    return out


def fill_adjoint(case, G, seed):
    """Bi-Maxwellian electrons (T_perp / T_par = 4) as rows of particle_t."""
    p = words(case["ppc"] * G.cells, 8)
    fill_thermal(p, G, case["ppc"], (0.05, 0.1, 0.1), seed, 10,
                 w=0.001 / case["ppc"])
    return p


# ---------------------------------------------------------------------------
# the framework's side
# ---------------------------------------------------------------------------

def simulation(case, seed, species=True, sort_interval=0):
    from vpic_amd import _lib, sim
    _lib.call("vpic_hip_init", 0)
    G = geo(case)
    s = sim.Simulation(G.grid())
    for k in range(2 if species else 0):
        name, q, m, _ = (ELECTRON, ION)[k]
        sp = sim.Species(name, q, m, case["ppc"] * G.cells, s.g,
                         sort_interval=sort_interval)
        fill_species(case, G, seed, k, sp.p.t.view(torch.float32).view(-1, 8))
        s.add_species(sp)
    return G, s


def f32(a, w):
    return a.t.view(torch.float32).view(-1, w)


def drifted(s, G, seed):
    """The species sorted, then moved on: what a diagnostic finds between
    two sorts."""
    for k, sp in enumerate(s.species):
        s.sort_p(sp)
        p = f32(sp.p, 8)
        p.copy_(drift_of(p, G, (ELECTRON, ION)[k][3], seed, 30 + k))


class Packed:
    """Device memory of an ensemble's packed array for torch.as_tensor, whose
    tensor keeps this object, and with it the ensemble, alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(
            shape=shape, typestr="<f4", data=(ptr, False), version=2)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        G, s = simulation(case, seed, sort_interval=case["steps"])
        if case["walls"]:
            sheet_fields(f32(s.fields, 20), G, seed)
        s.load_interpolator_array()
        return dict(case=case, sim=s)
    if kind == "push":
        G, s = simulation(case, seed, sort_interval=case["steps"])
        fill_fields(f32(s.fields, 20), G, 0.03, seed, TRACER_E)
        s.load_interpolator_array()
        return dict(case=case, sim=s)
    if kind == "vacuum":
        G, s = simulation(case, seed, species=False)
        fill_fields(f32(s.fields, 20), G, 0.1, seed)
        s.load_interpolator_array()
        return dict(case=case, sim=s)
    if kind in ("diag", "hydro"):
        G, s = simulation(case, seed, sort_interval=20)
        fill_fields(f32(s.fields, 20), G, 0.1, seed)
        s.load_interpolator_array()
        drifted(s, G, seed)
        return dict(case=case, sim=s)
    if kind == "collide":
        G, s = simulation(case, seed)
        drifted(s, G, seed)
        e, i = s.species
        s.takizuka_abe(e, i, 1e-3, 1, seed=seed % 1000)
        s.takizuka_abe(e, e, 1e-3, 1, seed=seed % 1000)
        s.step = 1
        return dict(case=case, sim=s)
    if kind == "ensemble":
        from vpic_amd import _lib, ensemble
        _lib.call("vpic_hip_init", 0)
        boxes = beam_boxes(case)
        geos = [Geo(nx, ny, 1, 0.5) for nx, ny, _, _ in boxes]
        nps = [p * G.cells for G, (_, _, p, _) in zip(geos, boxes)]
        e = ensemble.Ensemble([G.grid() for G in geos], nps)
        first = e.box(0)
        p = torch.as_tensor(Packed(e, first[0], (sum(nps), 8)), device=DEV)
        off = 0
        for b, (G, n, (_, _, ppc, drift)) in enumerate(zip(geos, nps, boxes)):
            fill_thermal(p[off:off + n], G, ppc, (0.01,) * 3, seed, 100 + b,
                         drift, 0.125 / ppc, True)
            off += n
        torch.cuda.synchronize()  # the ensemble works on its own stream
        e.prepare()
        nv = sum(G.nv for G in geos)
        views = [torch.as_tensor(Packed(e, ptr, (nv, w)), device=DEV)
                 for ptr, w in zip(first[1:], (20, 20, 12))]
        return dict(case=case, ens=e, views=views)
    G = geo(case)
    from vpic_amd import _lib
    _lib.call("vpic_hip_init", 0)
    p = fill_adjoint(case, G, seed)
    f = words(G.nv, 20)
    fill_fields(f, G, 0.02, seed)
    if case["bits"] == 64:
        f64 = torch.zeros((G.nv, 18), dtype=torch.float64, device=DEV)
        f64[:, :16] = f[:, :16].double()
        p, f = widen(p), f64
    return dict(case=case, p=p, f=f, g=G.grid())


def widen(p):
    """Rows of particle_t in the FP64 layout (the voxel in the fourth)."""
    q = torch.zeros(p.shape, dtype=torch.float64, device=DEV)
    q[:, 0:3] = p[:, 0:3].double()
    q.view(torch.int32)[:, 6] = p.view(torch.int32)[:, 3]
    q[:, 4:8] = p[:, 4:8].double()
    return q


# Particles of a step case are an output only while the sort's order is the
# same for every correct run: a last-bit difference of a current puts about
# one particle in 3e6 on the other side of a cell face after an interval, and
# the next sort then shifts every slot in between.  The push cases (given
# fields, so no feedback) return all of theirs at any size.
MOST_ORDERED = 100000


def particle_outputs(s):
    out = {}
    for sp in s.species:
        p = f32(sp.p, 8)
        out[sp.name] = dict(d=p[:, 0:3], i=p.view(torch.int32)[:, 3],
                            u=p[:, 4:7], w=p[:, 7])
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("step", "vacuum"):
        s = state["sim"]
        for _ in range(case["steps"]):
            s.advance()
        out = dict(fields=f32(s.fields, 20), interp=f32(s.interp, 20))
        if kind == "step":
            out["acc"] = f32(s.acc, 12)
            if sum(sp.np for sp in s.species) <= MOST_ORDERED:
                out.update(particle_outputs(s))
        return out
    if kind == "push":
        s = state["sim"]
        for sp in s.species:
            s.sort_p(sp)
        for _ in range(case["steps"]):
            s.clear_accumulator_array()
            s.advance_species()
            s.reduce_accumulator_array()
            s.step += 1
        return dict(acc=f32(s.acc, 12), **particle_outputs(s))
    if kind == "diag":
        s = state["sim"]
        en_f = s.energy_f()
        en_p = [s.energy_p(sp) for sp in s.species]
        rms = s.div_e_rms()
        return dict(fields=f32(s.fields, 20), en_f=en_f, en_p=en_p, rms=rms)
    if kind == "hydro":
        s = state["sim"]
        return {sp.name: s.hydro_moments(sp).view(np.float32).reshape(-1, 16)
                for sp in s.species}
    if kind == "collide":
        s = state["sim"]
        for op in s.collisions:
            op(s)
        s.step += 1
        return particle_outputs(s)
    if kind == "ensemble":
        state["ens"].step(case["steps"])
        return dict(zip(("fields", "interp", "acc"), state["views"]))
    from vpic_amd import adjoint
    w, u, d, f = adjoint.run(state["p"], state["f"], state["g"], -1.0, 1.0,
                             case["steps"], case["ckpt"], True, True, True)
    return dict(w=w, u=u, d=d, f=f)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

# per particle: the push reads and writes 32 B; a sort moves 32 B and reads
# its 4-B key.  Per voxel and step: cB twice and E (36 + 72 + 36 B), jf from
# the accumulator (72 B), the interpolator (96 B), the accumulator cleared
# and added to (48 + 96 B).  About 240 operations per particle and step.
PUSH_B, SORT_B, FIELD_B, ACC_B = 64, 68, 240, 216


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        n = c = 0
        for nx, ny, ppc, _ in beam_boxes(case):
            c += nx * ny
            n += nx * ny * ppc
        s = case["steps"]
        return dict(bytes=s * (PUSH_B * n + (FIELD_B + ACC_B) * c) +
                    SORT_B * n, flops=s * (240 * n + 150 * c))
    G = geo(case)
    c = G.cells
    if kind == "vacuum":
        return dict(bytes=case["steps"] * (FIELD_B + ACC_B) * c,
                    flops=case["steps"] * 120 * c)
    if kind == "adjoint":
        n, b = case["ppc"] * c, case["bits"] // 8
        s = case["steps"]
        # forward and recomputed steps, then the reverse: the particle read,
        # its adjoint (6 words) read and written, per cell the interpolator
        # and its adjoint, the accumulator adjoint and the fields
        return dict(bytes=b * s * (n * (2 * 16 + 8 + 12) + c * 2 * 114 +
                                   c * 120),
                    flops=s * (n * (2 * 240 + 900) + c * 500))
    n = 2 * case["ppc"] * c
    if kind == "step":
        s = case["steps"]
        return dict(bytes=s * (PUSH_B * n + (FIELD_B + ACC_B) * c) +
                    SORT_B * n, flops=s * (240 * n + 150 * c))
    if kind == "push":
        s = case["steps"]
        return dict(bytes=s * (PUSH_B * n + (72 + 144) * c) + SORT_B * n,
                    flops=s * 240 * n)
    if kind == "diag":
        # both energies and rho read the particles once each at most; the
        # field energies, the node sums and the error are per-voxel passes
        return dict(bytes=2 * 32 * n + c * (48 + 72 + 24 + 2 * 24),
                    flops=n * 60 + c * 60)
    if kind == "hydro":
        return dict(bytes=32 * n + 2 * c * (72 + 3 * 56), flops=n * 330)
    # the sorts of both species, the electrons scattered twice, the ions once
    return dict(bytes=SORT_B * n + 64 * (n // 2) * 3, flops=n * 300)


# About four times the largest differences seen.  A run of many steps parts
# from another by more than rounding: the interpolated force jumps where a
# particle crosses a face, so a last-bit difference that moves one crossing
# to another step changes that particle's momentum by a percent (32^3 cells,
# 2 x 64 per cell, 20 steps: 3 crossings moved, fields 1.6e-4 and currents
# 8.6e-4 from the 64-bit run; after one step 1.1e-7).
def tolerance(case):
    kind = case["kind"]
    if kind == "step":
        return {"rel": 5e-3, "max": 0.9, "differ": 1e-3}
    if kind == "vacuum":
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "push":
        return {"rel": 2e-5, "max": 1e-3, "differ": 1e-5}
    if kind in ("diag", "hydro"):
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "collide":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-5}
    if kind == "ensemble":
        return {"rel": 2e-3, "max": 0.5}
    if case["bits"] == 64:
        return {"rel": 1e-10, "max": 1e-7}
    return {"rel": 1e-3, "max": 0.5}


# ---------------------------------------------------------------------------
# the method in 64 bits
# ---------------------------------------------------------------------------

class Fields64:
    """E, cB, jf and tca as arrays [z, y, x], ghosts included; every update
    makes new arrays, so that torch can differentiate through it."""

    def __init__(self, G, f):
        self.G = G
        shape = [k + 2 for k in reversed(G.n)]
        v = f.double().view(*shape, -1)
        z = torch.zeros(shape, dtype=torch.float64, device=v.device)
        self.e = [v[..., k] for k in range(3)]
        self.b = [v[..., 4 + k] for k in range(3)]
        self.j = [z, z, z]
        self.t = [z, z, z]

    def part(self, lo, hi, shift=None):
        """Index of lo..hi per axis (x, y, z), moved by `shift`."""
        s = shift or (0, 0, 0)
        return tuple(slice(lo[k] + s[k], hi[k] + 1 + s[k])
                     for k in (2, 1, 0))

    def interpolators(self):
        n = self.G.n
        cut = lambda a, *s: a[self.part((1,) * 3, n, s)]  # noqa: E731
        unit = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
        out = []
        for c in range(3):
            y, z = unit[(c + 1) % 3], unit[(c + 2) % 3]
            yz = tuple(a + b for a, b in zip(y, z))
            w0, w1, w2, w3 = (cut(self.e[c], *s)
                              for s in ((0, 0, 0), y, z, yz))
            out += [0.25 * ((w3 + w0) + (w1 + w2)),
                    0.25 * ((w3 - w0) + (w1 - w2)),
                    0.25 * ((w3 - w0) - (w1 - w2)),
                    0.25 * ((w3 + w0) - (w1 + w2))]
        for c in range(3):
            w0, w1 = cut(self.b[c], 0, 0, 0), cut(self.b[c], *unit[c])
            out += [0.5 * (w1 + w0), 0.5 * (w1 - w0)]
        shape = [k + 2 for k in reversed(n)]
        full = torch.zeros(shape + [18], dtype=torch.float64,
                           device=self.e[0].device)
        full[self.part((1,) * 3, n)] = torch.stack(out, -1)
        return full.view(-1, 18)

    def coef(self, frac):
        G = self.G
        return [frac * G.dt * G.rd if k > 1 else 0.0 for k in G.n]

    def advance_b(self, frac):
        n, p, e = self.G.n, self.coef(frac), self.e
        b = []
        for c in range(3):
            y, z = (c + 1) % 3, (c + 2) % 3
            hi = [k for k in n]
            hi[c] += 1
            at = self.part((1,) * 3, hi)
            up = lambda a, k: a[self.part((1,) * 3, hi, [  # noqa: E731
                int(q == k) for q in range(3)])]
            new = self.b[c].clone()
            new[at] = self.b[c][at] - (p[y] * (up(e[z], y) - e[z][at]) -
                                       p[z] * (up(e[y], z) - e[y][at]))
            b.append(new)
        self.b = b

    def plane(self, x, k, lo, hi):
        """Index of plane k of axis x, lo..hi on the other two."""
        lo, hi = list(lo), list(hi)
        lo[x] = hi[x] = k
        return self.part(lo, hi)

    def ghosts(self):
        n = self.G.n
        b = [a.clone() for a in self.b]
        for x in range(3):
            wall = self.G.walls and x == 0
            for c in ((x + 1) % 3, (x + 2) % 3):
                hi = list(n)
                hi[c] += 1
                at = lambda k: self.plane(x, k, (1,) * 3, hi)  # noqa: E731
                first, last = b[c][at(1)].clone(), b[c][at(n[x])].clone()
                b[c] = b[c].clone()
                b[c][at(0)] = first if wall else last
                b[c][at(n[x] + 1)] = last if wall else first
        self.b = b

    def advance_e(self):
        self.ghosts()
        n, p, b, dt = self.G.n, self.coef(1.0), self.b, self.G.dt
        e, t = [], []
        for c in range(3):
            y, z = (c + 1) % 3, (c + 2) % 3
            hi = [k + 1 for k in n]
            hi[c] -= 1
            at = self.part((1,) * 3, hi)
            dn = lambda a, k: a[self.part((1,) * 3, hi, [  # noqa: E731
                -int(q == k) for q in range(3)])]
            curl = (p[y] * (b[z][at] - dn(b[z], y)) -
                    p[z] * (b[y][at] - dn(b[y], z)))
            tn, en = self.t[c].clone(), self.e[c].clone()
            tn[at] = curl
            en[at] = self.e[c][at] + (curl - dt * self.j[c][at])
            e.append(en)
            t.append(tn)
        if self.G.walls:
            for c in (1, 2):
                hi = [k + 1 for k in n]
                hi[c] -= 1
                for k in (1, n[0] + 1):
                    e[c][self.plane(0, k, (1,) * 3, hi)] = 0
                    t[c][self.plane(0, k, (1,) * 3, hi)] = 0
        self.e, self.t = e, t

    def current(self, acc):
        """jf from the accumulator (nv, 12): unload, walls, folds."""
        n, G = self.G.n, self.G
        a = acc.view(*[k + 2 for k in reversed(n)], 12)
        u = 0.25 * G.rd * G.rd / G.dt
        at = self.part((1,) * 3, [k + 1 for k in n])
        self.j = []
        for c in range(3):
            y, z = (c + 1) % 3, (c + 2) % 3
            back = lambda k, *axes: a[..., 4 * c + k][  # noqa: E731
                self.part((1,) * 3, [q + 1 for q in n],
                          [-int(q in axes) for q in range(3)])]
            j = torch.zeros_like(self.e[0])
            j[at] = u * (back(0) + back(1, y) + back(2, z) + back(3, y, z))
            self.j.append(j)
        for x in range(3):
            for c in ((x + 1) % 3, (x + 2) % 3):
                hi = [k + 1 for k in n]
                hi[c] -= 1
                lo_at = self.plane(x, 1, (1,) * 3, hi)
                hi_at = self.plane(x, n[x] + 1, (1,) * 3, hi)
                j = self.j[c].clone()
                if G.walls and x == 0:
                    j[lo_at] = 0
                    j[hi_at] = 0
                else:
                    s = j[lo_at] + j[hi_at]
                    j[lo_at] = s
                    j[hi_at] = s
                self.j[c] = j

    def step(self, acc):
        self.current(acc)
        self.advance_b(0.5)
        self.advance_e()
        self.advance_b(0.5)

    def out(self, width=20):
        z = torch.zeros_like(self.e[0])
        cols = list(self.e) + [z] + list(self.b) + [z] + list(self.t) + [z] \
            + list(self.j) + [z] * (width - 15)
        return torch.stack([c.reshape(-1) for c in cols], 1)


class Plasma64:
    """A species' positions, cells, momenta and weights in 64 bits."""

    def __init__(self, p, q, m):
        self.d = p[:, 0:3].double()
        self.i = p.view(torch.int32)[:, 3].long()
        self.u = p[:, 4:7].double()
        self.w = p[:, 7].double()
        self.q, self.m = q, m

    def sort(self):
        o = torch.sort(self.i, stable=True)[1]
        self.d, self.i, self.u, self.w = (a[o] for a in (self.d, self.i,
                                                         self.u, self.w))

    def out(self):
        return dict(d=self.d, i=self.i.int(), u=self.u, w=self.w)


def kick(f, d, u, qdt_2mc):
    """(half E impulse, cB) at the particles: f rows of interpolators."""
    x, y, z = d.unbind(1)
    h = torch.stack([(f[:, 0] + y * f[:, 1]) + z * (f[:, 2] + y * f[:, 3]),
                     (f[:, 4] + z * f[:, 5]) + x * (f[:, 6] + z * f[:, 7]),
                     (f[:, 8] + x * f[:, 9]) + y * (f[:, 10] + x * f[:, 11])],
                    1) * qdt_2mc
    b = torch.stack([f[:, 12] + x * f[:, 13], f[:, 14] + y * f[:, 15],
                     f[:, 16] + z * f[:, 17]], 1)
    return h, b


def rotate(u, b, v0):
    """Boris rotation with the quadratic-tangent correction."""
    v1 = (b * b).sum(1)
    v2 = v0 * v0 * v1
    v3 = v0 * (1 + v2 * (1 / 3 + v2 * 2 / 15))
    v4 = 2 * v3 / (1 + v1 * v3 * v3)
    w = u + v3[:, None] * torch.linalg.cross(u, b)
    return u + v4[:, None] * torch.linalg.cross(w, b)


def streaks(qw, s, mid):
    """The twelve quarter-face currents of a streak s about `mid`."""
    v5 = qw * s[:, 0] * s[:, 1] * s[:, 2] / 3
    out = []
    for c in range(3):
        my, mz = mid[:, (c + 1) % 3], mid[:, (c + 2) % 3]
        j = qw * s[:, c]
        out += [j * (1 - my) * (1 - mz) + v5, j * (1 + my) * (1 - mz) - v5,
                j * (1 - my) * (1 + mz) - v5, j * (1 + my) * (1 + mz) + v5]
    return torch.stack(out, 1)


def push64(G, d, i, u, w, q, m, fi, acc):
    """One push and deposit; returns (d, i, u, acc)."""
    h, b = kick(fi[i], d, u, q * G.dt / (2 * m))
    u = u + h
    v0 = (q * G.dt / (2 * m)) / torch.sqrt(1 + (u * u).sum(1))
    u = rotate(u, b, v0) + h
    s = u * (G.dt * G.rd) / torch.sqrt(1 + (u * u).sum(1))[:, None]
    qw = q * w
    end = d + 2 * s
    inside = (end.abs() <= 1).all(1)
    k = inside.nonzero()[:, 0]
    acc = acc.index_add(0, i[k], streaks(qw[k], s[k], d[k] + s[k]))
    out_d = torch.where(inside[:, None], end, d)
    out_i, out_u = i, u
    k = (~inside).nonzero()[:, 0]
    dk, ck, sk, uk = d[k], i[k], s[k], u[k]
    nx, ny, nz = G.n
    step = torch.tensor([1, nx + 2, (nx + 2) * (ny + 2)], device=d.device)
    size = torch.tensor(G.n, device=d.device)
    for _ in range(16):
        if not k.numel():
            break
        sgn = torch.where(sk > 0, 1.0, -1.0).to(sk.dtype)
        zero = sk == 0
        t = torch.where(zero, 3.4e38,
                        (sgn - dk) / torch.where(zero, 1.0, sk))
        tmin, axis = t.min(1)
        hit = tmin < 2
        seg = sk * (0.5 * torch.where(hit, tmin, 2.0))[:, None]
        acc = acc.index_add(0, ck, streaks(qw[k], seg, dk + seg))
        one = torch.nn.functional.one_hot(axis, 3).bool() & hit[:, None]
        dk = torch.where(one, sgn, dk + 2 * seg)
        sk = sk - seg
        # the neighbour through that face
        c = torch.stack([ck % (nx + 2), (ck // (nx + 2)) % (ny + 2),
                         ck // ((nx + 2) * (ny + 2))], 1)
        up = sgn > 0
        edge = torch.where(up, c == size, c == 1)
        move = torch.where(up, 1, -1) * torch.where(edge, 1 - size, 1)
        if G.walls:
            back = one & edge & torch.tensor([True, False, False],
                                             device=d.device)
            uk = torch.where(back, -uk, uk)
            sk = torch.where(back, -sk, sk)
            one = one & ~back
        ck = ck + (move * step * one).sum(1)
        dk = torch.where(one, -sgn, dk)
        done = (~hit).nonzero()[:, 0]
        at = k[done]
        out_d = out_d.index_copy(0, at, dk[done])
        out_i = out_i.index_copy(0, at, ck[done])
        out_u = out_u.index_copy(0, at, uk[done])
        go = hit.nonzero()[:, 0]
        k, dk, ck, sk, uk = k[go], dk[go], ck[go], sk[go], uk[go]
    return out_d, out_i, out_u, acc


def push_all(G, species, fi):
    acc = torch.zeros((G.nv, 12), dtype=torch.float64, device=DEV)
    for p in species:
        n = p.d.shape[0]
        got = [push64(G, p.d[a:a + CHUNK], p.i[a:a + CHUNK], p.u[a:a + CHUNK],
                      p.w[a:a + CHUNK], p.q, p.m, fi, acc)
               for a in range(0, min(n, CHUNK), CHUNK)]
        for a in range(CHUNK, n, CHUNK):
            got.append(push64(G, p.d[a:a + CHUNK], p.i[a:a + CHUNK],
                              p.u[a:a + CHUNK], p.w[a:a + CHUNK], p.q, p.m,
                              fi, got[-1][3]))
        p.d, p.i, p.u = (torch.cat([g[k] for g in got]) for k in range(3))
        acc = got[-1][3]
    return acc


def pad(fi):
    return torch.cat([fi, torch.zeros_like(fi[:, :2])], 1)


def species64(case, G, seed, both=(0, 1)):
    out = []
    for k in both:
        p = words(case["ppc"] * G.cells, 8)
        fill_species(case, G, seed, k, p)
        out.append((p, (ELECTRON, ION)[k]))
    return out


def run64(G, f, species, steps):
    """The step loop: (fields, interpolators, last accumulator)."""
    F = Fields64(G, f)
    fi = F.interpolators()
    acc = torch.zeros((G.nv, 12), dtype=torch.float64, device=DEV)
    for _ in range(steps):
        acc = push_all(G, species, fi)
        F.step(acc)
        fi = F.interpolators()
    return F, fi, acc


# Particle steps of a run whose fields act back on the particles, for which
# the 64-bit values say something about a 32-bit run: past it some crossing
# has moved to another step (see tolerance), in one correct run as in
# another, and the distance from the 64-bit run is that crossing's.
MOST_SAME_PATH = 4000000
MOST_64 = 1000000000  # particle steps: about 20 s


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "ensemble":
            return exact_ensemble(case, seed)
        G = geo(case)
        if kind == "vacuum":
            f = words(G.nv, 20)
            fill_fields(f, G, 0.1, seed)
            F, fi, _ = run64(G, f, [], case["steps"])
            return dict(fields=F.out(), interp=pad(fi))
        if kind == "adjoint":
            n = case["ppc"] * G.cells * case["steps"]
            if n > (MOST_SAME_PATH if case["bits"] == 32 else MOST_64 // 5):
                return None
            with torch.enable_grad():
                return exact_adjoint(case, G, seed)
        n = 2 * case["ppc"] * G.cells * case.get("steps", 1)
        if n > (MOST_SAME_PATH if kind == "step" else MOST_64):
            return None
        if kind == "step":
            f = torch.zeros((G.nv, 20), device=DEV)
            if case["walls"]:
                sheet_fields(f, G, seed)
            sp = [Plasma64(p, s[1], s[2]) for p, s in
                  species64(case, G, seed)]
            for p in sp:
                p.sort()
            F, fi, acc = run64(G, f, sp, case["steps"])
            out = dict(fields=F.out(), interp=pad(fi), acc=acc)
            if sum(p.w.numel() for p in sp) <= MOST_ORDERED:
                out.update(electron=sp[0].out(), ion=sp[1].out())
            return out
        if kind == "push":
            f = words(G.nv, 20)
            fill_fields(f, G, 0.03, seed, TRACER_E)
            fi = Fields64(G, f).interpolators()
            sp = [Plasma64(p, s[1], s[2]) for p, s in
                  species64(case, G, seed)]
            for p in sp:
                p.sort()
            for _ in range(case["steps"]):
                acc = push_all(G, sp, fi)
            return dict(acc=acc, electron=sp[0].out(), ion=sp[1].out())
        sp = []
        for k, (p, s) in enumerate(species64(case, G, seed)):
            sp.append(Plasma64(drift_of(p, G, s[3], seed, 30 + k), s[1],
                               s[2]))
        if kind == "collide":
            return exact_collide(case, G, seed, sp)
        f = words(G.nv, 20)
        fill_fields(f, G, 0.1, seed)
        F = Fields64(G, f)
        fi = F.interpolators()
        if kind == "diag":
            return exact_diag(G, F, f, sp, fi)
        return {name: exact_hydro(G, p, fi)
                for name, p in zip(("electron", "ion"), sp)}


def weights(d):
    """Trilinear weights of the 8 nodes (x fastest), times 8."""
    out = []
    for k in range(8):
        s = [1 + (1 if k >> a & 1 else -1) * d[:, a] for a in range(3)]
        out.append(s[0] * s[1] * s[2])
    return torch.stack(out, 1)


def nodes(G, i):
    sy, sz = G.n[0] + 2, (G.n[0] + 2) * (G.n[1] + 2)
    off = torch.tensor([(k & 1) + (k >> 1 & 1) * sy + (k >> 2) * sz
                        for k in range(8)], device=DEV)
    return i[:, None] + off


def fold_nodes(G, a):
    """Periodic node planes summed, axis by axis; a: [z, y, x, ...]."""
    for x, dim in ((0, 2), (1, 1), (2, 0)):
        n = G.n[x]
        box = [slice(1, k + 2) for k in reversed(G.n)]
        lo, hi = list(box), list(box)
        lo[dim], hi[dim] = slice(1, 2), slice(n + 1, n + 2)
        s = a[tuple(lo)] + a[tuple(hi)]
        a[tuple(lo)] = s
        a[tuple(hi)] = s
    return a


def exact_diag(G, F, f, sp, fi):
    n = G.n
    rho = torch.zeros(G.nv, dtype=torch.float64, device=DEV)
    en_p = []
    for p in sp:
        q = p.q * G.r8V * p.w[:, None] * weights(p.d)
        rho.index_add_(0, nodes(G, p.i).reshape(-1), q.reshape(-1))
        h, _ = kick(fi[p.i], p.d, p.u, p.q * G.dt / (2 * p.m))
        u2 = ((p.u + h) ** 2).sum(1)
        en_p.append(float((p.m * p.w * u2 / (1 + torch.sqrt(1 + u2))).sum()))
    shape = [k + 2 for k in reversed(n)]
    rho = fold_nodes(G, rho.view(*shape, 1))[..., 0]
    unit = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
    cut = lambda a, *s: a[F.part((1,) * 3, n, s)]  # noqa: E731
    en_f = []
    for c in range(3):
        y, z = unit[(c + 1) % 3], unit[(c + 2) % 3]
        yz = tuple(a + b for a, b in zip(y, z))
        en_f.append(0.25 * sum((cut(F.e[c], *s) ** 2).sum()
                               for s in ((0, 0, 0), y, z, yz)))
    for c in range(3):
        en_f.append(0.5 * sum((cut(F.b[c], *s) ** 2).sum()
                              for s in ((0, 0, 0), unit[c])))
    en_f = 0.5 * G.dV * torch.stack(en_f)
    # normal-E ghosts, then div E - rho on the nodes
    e = [a.clone() for a in F.e]
    for x in range(3):
        hi = [k + 1 for k in n]
        at = lambda k: F.plane(x, k, (1,) * 3, hi)  # noqa: E731
        first, last = e[x][at(1)].clone(), e[x][at(n[x])].clone()
        e[x][at(0)], e[x][at(n[x] + 1)] = last, first
    hi = [k + 1 for k in n]
    at = F.part((1,) * 3, hi)
    err = -rho[at]
    for c in range(3):
        if n[c] > 1:
            dn = e[c][F.part((1,) * 3, hi, [-k for k in unit[c]])]
            err = err + G.rd * (e[c][at] - dn)
    wt = torch.ones_like(err)
    for dim in range(3):
        for k in (0, -1):
            wt.select(dim, k).mul_(0.5)
    rms = math.sqrt(float((wt * err ** 2).sum()) / G.cells)
    out = f.double().view(*shape, 20).clone()
    for c in range(3):
        out[..., c] = e[c]
    out[..., 15] = rho
    out[at + (3,)] = err
    return dict(fields=out.view(-1, 20), en_f=en_f, en_p=en_p, rms=rms)


def exact_hydro(G, p, fi):
    q2m = p.q * G.dt / (2 * p.m)
    h, b = kick(fi[p.i], p.d, p.u, q2m)
    u = p.u + h
    u2 = (u * u).sum(1)
    g = torch.sqrt(1 + u2)
    ke = u2 / (1 + g)
    v0 = (q2m / 2) / g
    w1 = (b * b).sum(1)
    w2 = v0 * v0 * w1
    w3 = v0 * (1 + w2 / 3 * (1 + 0.4 * w2))
    w4 = 2 * w3 / (1 + w1 * w3 * w3)
    w = u + w3[:, None] * torch.linalg.cross(u, b)
    u = u + w4[:, None] * torch.linalg.cross(w, b)
    v = u / g[:, None]
    mom = torch.stack([v[:, 0] * p.q, v[:, 1] * p.q, v[:, 2] * p.q,
                       torch.full_like(g, p.q)] +
                      [p.m * c for c in (u[:, 0], u[:, 1], u[:, 2], ke,
                                         u[:, 0] * v[:, 0],
                                         u[:, 1] * v[:, 1],
                                         u[:, 2] * v[:, 2],
                                         u[:, 1] * v[:, 2],
                                         u[:, 2] * v[:, 0],
                                         u[:, 0] * v[:, 1])], 1)
    wn = G.r8V * p.w[:, None] * weights(p.d)
    at = nodes(G, p.i)
    out = torch.zeros((G.nv, 16), dtype=torch.float64, device=DEV)
    for k in range(8):
        out[:, :14].index_add_(0, at[:, k], wn[:, k:k + 1] * mom)
    shape = [k + 2 for k in reversed(G.n)]
    return fold_nodes(G, out.view(*shape, 16)).view(-1, 16)


def exact_ensemble(case, seed):
    parts = []
    boxes = beam_boxes(case)
    total = sum(nx * ny * ppc for nx, ny, ppc, _ in boxes) * case["steps"]
    if total > MOST_SAME_PATH:
        return None
    for b, (nx, ny, ppc, drift) in enumerate(boxes):
        G = Geo(nx, ny, 1, 0.5)
        p = words(ppc * G.cells, 8)
        fill_thermal(p, G, ppc, (0.01,) * 3, seed, 100 + b, drift,
                     0.125 / ppc, True)
        F, fi, acc = run64(G, torch.zeros((G.nv, 20), device=DEV),
                           [Plasma64(p, -1.0, 1.0)], case["steps"])
        parts.append((F.out(), pad(fi), acc))
    return dict(zip(("fields", "interp", "acc"),
                    (torch.cat([x[k] for x in parts]) for k in range(3))))


def exact_adjoint(case, G, seed):
    from torch.utils.checkpoint import checkpoint
    p32 = fill_adjoint(case, G, seed)
    f = words(G.nv, 20)
    fill_fields(f, G, 0.02, seed)
    p = Plasma64(p32, -1.0, 1.0)
    d0 = d = p.d.clone().requires_grad_()
    u0 = u = p.u.clone().requires_grad_()
    f0 = f[:, [0, 1, 2, 4, 5, 6]].double().requires_grad_()
    shape = [k + 2 for k in reversed(G.n)]
    zero = torch.zeros(G.nv, dtype=torch.float64, device=DEV)
    i = p.i

    def one(d, u, i, *c):
        F = Fields64(G, torch.zeros((G.nv, 20), device=DEV))
        F.e, F.b = [a.view(shape) for a in c[:3]], \
            [a.view(shape) for a in c[3:]]
        acc = torch.zeros((G.nv, 12), dtype=torch.float64, device=DEV)
        d, i, u, acc = push64(G, d, i, u, p.w, -1.0, 1.0, F.interpolators(),
                              acc)
        F.step(acc)
        return (d, u, i, *[a.reshape(-1) for a in F.e + F.b])

    state = (d, u, i, *f0.unbind(1))
    for _ in range(case["steps"]):
        state = checkpoint(one, *state, use_reentrant=False)
    F = Fields64(G, torch.zeros((G.nv, 20), device=DEV))
    unit = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
    w = zero.sum()
    for c in range(3):
        b = state[6 + c].view(shape)
        for s in ((0, 0, 0), unit[c]):
            w = w + 0.5 * (b[F.part((1,) * 3, G.n, s)] ** 2).sum()
    w = 0.5 * G.dV * w
    gd, gu, gf = torch.autograd.grad(w, (d0, u0, f0))
    return dict(w=float(w.detach()), u=gu, d=gd, f=gf)


# -- collisions: the counter-based stream, the shuffle and the pairing --------

MASK = 0xFFFFFFFF


def philox(ctr0, voxel, call, key):
    """Philox4x32-10 words of counter {ctr0, voxel, call} (Salmon et al.,
    SC'11), as int64 tensors [4, ...]."""
    c = [ctr0, voxel, torch.full_like(ctr0, call & MASK),
         torch.full_like(ctr0, call >> 32)]
    k0, k1 = key & MASK, key >> 32

    def mul(m, a):  # 32 x 32 bits to (high, low) within int64
        p, q = m * (a & 0xFFFF), m * (a >> 16)
        t = q + (p >> 16)
        return t >> 16, (t & 0xFFFF) << 16 | (p & 0xFFFF)

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & MASK, (k1 + 0xBB67AE85) & MASK
    return torch.stack(c)


def operator_key(seed, index):
    """The key of a simulation's collision operator `index` for a seed (the
    splitmix64 finaliser of both)."""
    m = (1 << 64) - 1
    z = ((int(seed) << 16) + int(index) + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


class Stream:
    """Each voxel's own stream: the next word, for the voxels asked."""

    def __init__(self, vox, call, key):
        self.vox, self.call, self.key = vox, call, key
        self.n = torch.zeros_like(vox)

    def u32(self, on):
        w = philox(self.n >> 2, self.vox, self.call, self.key)
        out = w.gather(0, (self.n & 3)[None])[0]
        self.n = self.n + on.long()
        return out


def collide64(a, b, mu_a, mu_b, std, rng, on, ia, ib):
    """One collision per voxel where `on`, between rows ia of a and ib of
    b."""
    du = a.u[ia] - b.u[ib]
    sq = (du * du).float()  # the axis is chosen by the 32-bit squares
    d0 = torch.zeros_like(ia)
    t1 = sq[:, 0]
    d0 = torch.where(sq[:, 1] < t1, 1, d0)
    t1 = torch.minimum(sq[:, 1], t1)
    d0 = torch.where(sq[:, 2] < t1, 2, d0)
    ur = torch.sqrt((du * du).sum(1))
    d1, d2 = (d0 + 1) % 3, (d0 + 2) % 3
    c1, c2 = du.gather(1, d1[:, None])[:, 0], du.gather(1, d2[:, None])[:, 0]
    t0 = 1 / torch.sqrt(c1 * c1 + c2 * c2 + 1.1754943508222875e-38)
    t = torch.zeros_like(du)
    t.scatter_(1, d1[:, None], (t0 * c2)[:, None])
    t.scatter_(1, d2[:, None], (-t0 * c1)[:, None])
    r24 = 1.0 / 16777216.0
    u1 = ((rng.u32(on) >> 8).double() + 1) * r24
    u2 = (rng.u32(on) >> 8).double() * r24
    dd = torch.minimum(std / torch.sqrt(ur) / ur, torch.ones_like(ur)) * \
        torch.sqrt(-2 * torch.log(u1)) * torch.cos(2 * math.pi * u2)
    t0 = 2 * dd / (1 + dd * dd)
    th = 2 * math.pi * (rng.u32(on) >> 8).double() * r24
    s = (-dd * t0)[:, None] * du + (t0 * ur * torch.cos(th))[:, None] * t + \
        (t0 * torch.sin(th))[:, None] * torch.linalg.cross(du, t)
    pick = (rng.u32(on) >> 8).double() * r24
    wa, wb = a.w[ia], b.w[ib]
    ma = torch.where((wb < wa) & (wa * pick > wb), 0.0, mu_a)
    mb = torch.where((wa < wb) & (wb * pick > wa), 0.0, mu_b)
    o = on.nonzero()[:, 0]
    a.u[ia[o]] = (a.u[ia] + ma[:, None] * s)[o]
    b.u[ib[o]] = (b.u[ib] - mb[:, None] * s)[o]


def operator64(G, a, b, cvar0, key, call):
    """One application of the operator to sorted species a and b."""
    same = a is b
    edges = torch.arange(G.nv + 1, device=DEV)
    pa = torch.searchsorted(a.i, edges)
    pb = torch.searchsorted(b.i, edges)
    vox = ((pa[1:] - pa[:-1]) > 0).nonzero()[:, 0]
    k0, nk = pa[vox], (pa[1:] - pa[:-1])[vox]
    rng = Stream(vox, call, key)
    order = torch.arange(a.i.numel(), device=DEV)
    dens = torch.zeros(vox.shape, dtype=torch.float64, device=DEV)
    for i in range(int(nk.max()) - 1):
        on = i < nk - 1
        left = (nk - i).clamp(min=1)
        rn = MASK // left
        need, j = on.clone(), torch.zeros_like(nk)
        while bool(need.any()):
            got = rng.u32(need) // rn
            j = torch.where(need, got, j)
            need = need & (got >= left)
        s, t = (k0 + i)[on], (k0 + i + j)[on]
        order[s], order[t] = order[t], order[s]
    a.d, a.i, a.u, a.w = a.d[order], a.i[order], a.u[order], a.w[order]
    dens.index_add_(0, torch.repeat_interleave(
        torch.arange(vox.numel(), device=DEV), nk), a.w)
    mu = a.m * b.m / (a.m + b.m)
    mu_a, mu_b = b.m / (a.m + b.m), a.m / (a.m + b.m)
    cvar = cvar0 * (a.q * a.q * b.q * b.q) / (mu * mu)
    tv = G.dt / G.dV
    if same:
        odd = (nk % 2 == 1) & (nk >= 3)
        std = torch.sqrt(0.5 * dens * cvar * tv)
        for x, y in ((0, 1), (0, 2), (1, 2)):
            on = odd
            ia = torch.where(on, k0 + x, 0 * k0)
            ib = torch.where(on, k0 + y, 0 * k0)
            collide64(a, b, mu_a, mu_b, std, rng, on, ia, ib)
        nk = torch.where(odd, nk - 3, nk)
        k0 = torch.where(odd, k0 + 3, k0)
        nk = nk // 2
        nl, l0 = nk, k0 + nk
        std = torch.sqrt(cvar * dens * tv)
    else:
        l0, nl = pb[vox], (pb[1:] - pb[:-1])[vox]
        dl = torch.zeros(G.nv, dtype=torch.float64, device=DEV)
        dl.index_add_(0, b.i, b.w)
        std = torch.sqrt(cvar * torch.minimum(dl[vox], dens) * tv)
    live = (nk > 0) & (nl > 0)
    big, small = torch.maximum(nk, nl), torch.minimum(nk, nl).clamp(min=1)
    ii = big // small
    rem = big - ii * small
    for s in range(int(big.max())):
        on = live & (s < big)
        first = rem * (ii + 1)
        grp = torch.where(s < first, s // (ii + 1),
                          rem + (s - first) // ii.clamp(min=1))
        many = torch.full_like(nk, s)
        ks = torch.where(nk > nl, many, grp)
        ls = torch.where(nk > nl, grp, many)
        ia = torch.where(on, k0 + ks, 0 * k0)
        ib = torch.where(on, l0 + ls, 0 * l0)
        collide64(a, b, mu_a, mu_b, std, rng, on, ia, ib)


def exact_collide(case, G, seed, sp):
    e, i = sp
    for p in sp:
        p.sort()
    key = seed % 1000
    operator64(G, e, i, 1e-3, operator_key(key, 0), 1)
    operator64(G, e, e, 1e-3, operator_key(key, 1), 1)
    return dict(electron=e.out(), ion=i.out())
