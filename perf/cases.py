"""The workloads whose speed is tracked, and what they compute.

A case is a stretch of a simulation as a program runs it between two
outputs: the context with its mesh and initial state is set up once
(`prepare`), then `run` advances a number of steps and downloads the whole
conserved state, as the main loop does before it writes a file.  The cases
cover both physics (hydro, MHD), the three numerical forms, uniform and
refined meshes, radiative cooling, wind sources and mesh changes, from 8
blocks (where launches and latency count) to 4096 (where throughput does).

`exact` advances the same initial state with the same scheme in 64 bits in
plain torch, without the package: the discretisation of the Godunov update
(first-order predictor over dt/2, limited second-order corrector over dt,
viscosity, cooling), the face exchange between refinement levels, and the
start-up ramp of the timestep.
"""
import math

import numpy as np
import torch

NC = 16                      # cells per block edge
NB = 20                      # with two ghost layers
PC, AMU, KB = 3.085677588e+18, 1.660538782e-24, 1.380650400e-16
PI_REF = 3.14159265358979
MU0, MUI = 1.3, 0.61

CASES = (
    # the smallest mesh of the test suite: one MHD box of 32^3 with walls,
    # open and periodic sides; every launch leaves most of the chip idle
    dict(name="mhd_box_8", ic="ot", form="fused32", solver="hlle", limiter="superbee", visc=2.0e-3, bc="frppff",
         nx=1, ny=1, nz=1, base=2, steps=50),
    # a shock tube: 32 blocks in a row, 512 x 16 x 16 cells
    dict(name="shock_tube_32", ic="shock", form="fused32", solver="hlld", limiter="minmod", visc=0.0, bc="ffffff",
         nx=32, ny=1, nz=1, base=1, steps=50),
    # a parameter study's resolution: periodic MHD turbulence at 64^3
    dict(name="mhd_vortex_64", ic="ot", form="fused32", solver="hlld", limiter="minmod", visc=0.0, bc="pppppp",
         nx=1, ny=1, nz=1, base=3, steps=50),
    # the production resolution of the headline benchmark, 4096 blocks
    dict(name="mhd_vortex_4096", ic="ot", form="fused32", solver="hlld", limiter="minmod", visc=0.0, bc="pppppp",
         nx=1, ny=1, nz=1, base=5, steps=48),
    # the precision reference of the fused kernels on a box of odd extents
    dict(name="mhd_vortex_fp64_240", ic="ot", form="fused64", solver="hlld", limiter="minmod", visc=0.0,
         bc="pppppp", nx=5, ny=3, nz=2, base=2, steps=20),
    # a point explosion at 64^3 with viscosity, the hydro parameter study
    dict(name="blast_64", ic="blast", form="fused32", solver="hllc", limiter="minmod", visc=5.0e-3, bc="ffffff",
         nx=1, ny=1, nz=1, base=3, steps=50),
    # the same at production size, 12^3 blocks
    dict(name="blast_1728", ic="blast", form="fused32", solver="hllc", limiter="minmod", visc=5.0e-3, bc="ffffff",
         nx=3, ny=3, nz=3, base=3, steps=24),
    # a supernova remnant in a clumpy, radiatively cooling medium on 4 levels
    dict(name="remnant_amr", ic="clumps", form="fused32", solver="hllc", limiter="minmod", visc=5.0e-3,
         bc="ffffff", nx=1, ny=1, nz=1, base=3, levels=4, radius=0.30, cooling=True, steps=24),
    # stellar winds on 3 levels with a mesh change every few steps: flags from
    # the gradients, the finer region grown, later shrunk again
    dict(name="winds_regrid", ic="winds", form="fused32", solver="hll", limiter="minmod", visc=5.0e-3, bc="ffffff",
         nx=1, ny=1, nz=1, base=3, levels=3, radius=0.24, cooling=True, steps=16, regrid=True),
    # the default form (the reference's arithmetic), hydro at 64^3
    dict(name="blast_plain_64", ic="blast", form="plain", solver="hllc", limiter="minmod", visc=5.0e-3, bc="ffffff",
         nx=1, ny=1, nz=1, base=3, steps=20),
    # the default form, MHD at 128^3
    dict(name="mhd_vortex_plain_512", ic="ot", form="plain", solver="hlld", limiter="minmod", visc=0.0, bc="pppppp",
         nx=1, ny=1, nz=1, base=4, steps=10),
    # the default form on 3 levels with cooling and reflecting floor
    dict(name="remnant_plain_amr", ic="clumps", form="plain", solver="hll", limiter="vanleer", visc=5.0e-3,
         bc="ffffrf", nx=1, ny=1, nz=1, base=3, levels=3, radius=0.26, cooling=True, steps=10),
)


def listed():
    return [dict(c) for c in CASES]


def draw(rng):
    """One more case: any physics, form, solver, limiter and boundary that
    the listed ones stand for, on 8 to about 1500 blocks."""
    mhd = rng.random() < 0.5
    form = rng.choice(("fused32", "fused32", "fused32", "fused64", "plain", "plain"))
    c = dict(form=form, limiter=rng.choice(("minmod", "minmod", "vanleer", "woodward", "superbee")))
    refined = rng.random() < 0.35
    # extents in root blocks, odd ones among them, at one or two base levels
    base = 2
    want = 2.0 ** rng.uniform(3.0, 10.5) / 8.0
    if refined:
        want = 2.0 ** rng.uniform(3.0, 6.5) / 8.0
    n = [1, 1, 1]
    while n[0] * n[1] * n[2] < want:
        n[rng.randrange(3)] += 1
    c.update(nx=n[0], ny=n[1], nz=n[2], base=base)
    if mhd:
        c.update(ic="ot", solver=rng.choice(("hlld", "hlld", "hlle")), visc=rng.choice((0.0, 0.0, 2.0e-3)))
        c["bc"] = "pppppp" if not refined and rng.random() < 0.6 else "ffffff"
    else:
        c.update(ic=rng.choice(("blast", "clumps", "winds")) if refined else "blast",
                 solver=rng.choice(("hllc", "hll")), visc=5.0e-3, bc=rng.choice(("ffffff", "rrrrrr", "ffffrf")))
        if c["ic"] != "blast":
            c["cooling"] = rng.random() < 0.7
    if refined:
        c.update(levels=rng.choice((2, 3)), radius=rng.uniform(0.15, 0.3))
    blocks = len(_mesh(c))
    budget = {"fused32": 24000, "fused64": 8000, "plain": 3000}[form]
    c["steps"] = int(max(4, min(50, budget // blocks)))
    return c


# ---------------------------------------------------------------------------
# Meshes: octree leaves (level, x, y, z), 0-based coordinates per level
# ---------------------------------------------------------------------------
def _dims(c, level):
    f = 1 << (level - 1)
    return (c["nx"] * f, c["ny"] * f, c["nz"] * f)


def _centres(c):
    """Refinement and source centres, as fractions of the box's edges."""
    if c["ic"] == "winds":
        return ((0.31, 0.62, 0.44), (0.66, 0.37, 0.58), (0.52, 0.71, 0.69))
    return ((0.5, 0.5, 0.5),)


def _mesh(c, grow=1.0):
    """The active blocks, finest region within `radius` of a centre on the
    first refined level and about half of that on each level above; face
    neighbours differ by one level at most."""
    base, top = c["base"], c["base"] + c.get("levels", 1) - 1
    refined = {l: set() for l in range(0, top + 1)}
    for l in range(1, base):
        n = _dims(c, l)
        refined[l] = {(x, y, z) for z in range(n[2]) for y in range(n[1]) for x in range(n[0])}
    r = c.get("radius", 0.0) * grow
    for l in range(base, top):
        n = _dims(c, l)
        small = min(n)
        for cen in _centres(c):
            lo = [max(0, int((cen[d] * n[d]) - r * small) - 1) for d in range(3)]
            hi = [min(n[d] - 1, int((cen[d] * n[d]) + r * small) + 1) for d in range(3)]
            for z in range(lo[2], hi[2] + 1):
                for y in range(lo[1], hi[1] + 1):
                    for x in range(lo[0], hi[0] + 1):
                        d2 = 0.0
                        for d, q in enumerate((x, y, z)):
                            p = cen[d] * n[d]
                            near = min(max(p, q), q + 1)
                            d2 += ((near - p) / small) ** 2
                        if d2 <= r * r and (l == base or (x >> 1, y >> 1, z >> 1) in refined[l - 1]):
                            refined[l].add((x, y, z))
        r *= 0.55
    for l in range(top - 1, 1, -1):
        n = _dims(c, l)
        for x, y, z in list(refined[l]):
            refined[l - 1].add((x >> 1, y >> 1, z >> 1))
            for d in range(3):
                for s in (-1, 1):
                    p = [x, y, z]
                    p[d] += s
                    if 0 <= p[d] < n[d]:
                        refined[l - 1].add((p[0] >> 1, p[1] >> 1, p[2] >> 1))
    out = []
    n = _dims(c, 1)
    nodes = [(x, y, z) for z in range(n[2]) for y in range(n[1]) for x in range(n[0])]
    for l in range(1, top + 1):
        nxt = []
        for p in nodes:
            if p in refined[l]:
                nxt += [(2 * p[0] + i, 2 * p[1] + j, 2 * p[2] + k) for k in (0, 1) for j in (0, 1) for i in (0, 1)]
            else:
                out.append((l,) + p)
        nodes = nxt
    return out


def _block_ids(c, mesh):
    """The solver's block numbers: level by level, x fastest."""
    first = [1]
    for l in range(1, 16):
        n = _dims(c, l)
        first.append(first[-1] + n[0] * n[1] * n[2])
    out = []
    for l, x, y, z in mesh:
        n = _dims(c, l)
        out.append(first[l - 1] + x + y * n[0] + z * n[0] * n[1])
    return np.asarray(out, dtype=np.int32)


# ---------------------------------------------------------------------------
# Physics and units of a case
# ---------------------------------------------------------------------------
def _units(c):
    """Code units in cgs: length, density, velocity."""
    if c["ic"] in ("clumps", "winds"):
        return PC, MU0 * AMU, 1.0e5
    return 1.0, 1.0, 1.0


def _gamma(c):
    return 2.0 if c["ic"] == "shock" else 5.0 / 3.0


def _phys(c):
    """Edge lengths of the box in cgs: cubic cells."""
    edge = 20.0 * PC if c["ic"] in ("clumps", "winds") else 1.0
    n = (c["nx"], c["ny"], c["nz"])
    return tuple(edge * q / max(n) for q in n)


def _dx(c, level):
    p, l_sc = _phys(c), _units(c)[0]
    return [p[d] / (NC * (c["nx"], c["ny"], c["nz"])[d] * 2.0 ** (level - 1)) / l_sc for d in range(3)]


def _top(c):
    return c["base"] + c.get("levels", 1) - 1


def _winds(c):
    """(x, y, z, radius, mass loss, speed, temperature, mu) of each source in
    cgs: 100 cm^-3 and 300 km/s at a radius of 4 finest cells."""
    if c["ic"] != "winds":
        return []
    p, r = _phys(c), 4.0 * _dx(c, _top(c))[0] * PC
    rho, v = 100.0 * MU0 * AMU, 3.0e7
    return [(q[0] * p[0], q[1] * p[1], q[2] * p[2], r, rho * v * r * r * 4.0 * math.pi, v, 1.2e4, MU0)
            for q in _centres(c)]


def _table():
    """A smooth log-log cooling curve, logT 4..8 (erg cm^3 s^-1)."""
    t = 4.0 + 4.0 * np.arange(100) / 99.0
    x = (t - 4.0) / 4.0
    return t, -22.0 + 0.8 * np.sin(np.pi * x) + 0.3 * np.exp(-((t - 5.2) ** 2) / 0.1) - 0.2 * np.exp(
        -((t - 6.9) ** 2) / 0.1)


def _initial(c, mesh, seed):
    """Conserved state [block][variable][16][16][16] from the seed."""
    rng = np.random.default_rng(seed)
    nb, g = len(mesh), _gamma(c)
    l_sc, d_sc, v_sc = _units(c)
    lev = np.array([m[0] for m in mesh])
    dxs = np.array([_dx(c, l) for l in range(1, _top(c) + 1)])[lev - 1]
    cell = np.arange(NC) + 0.5
    org = np.array([m[1:] for m in mesh], dtype=np.float64) * NC
    axis = [((org[:, d, None] + cell[None, :]) * dxs[:, d, None]) for d in range(3)]      # [nb][16], code units
    X, Y, Z = axis[0][:, None, None, :], axis[1][:, None, :, None], axis[2][:, :, None, None]
    box = [p / l_sc for p in _phys(c)]
    full = (nb, NC, NC, NC)
    mhd = c["ic"] in ("ot", "shock")
    U = np.zeros((nb, 8 if mhd else 5) + full[1:])
    if c["ic"] == "ot":
        # Orszag-Tang vortex with seeded phases and amplitudes, and noise along z
        a = 1.0 + 0.1 * rng.uniform(-1, 1, 4)
        ph = rng.uniform(0.0, 2.0 * math.pi, 4)
        kx, ky = 2.0 * math.pi / box[0], 2.0 * math.pi / box[1]
        rho, p, b0 = 25.0 / (36.0 * math.pi), 5.0 / (12.0 * math.pi), 1.0 / math.sqrt(4.0 * math.pi)
        vx, vy = -a[0] * np.sin(ky * Y + ph[0]), a[1] * np.sin(kx * X + ph[1])
        vz = 1.0e-2 * rng.uniform(-1, 1, full)
        bx, by = -a[2] * b0 * np.sin(ky * Y + ph[2]), a[3] * b0 * np.sin(2.0 * kx * X + ph[3])
        U[:, 0] = rho
        U[:, 1] = rho * vx
        U[:, 2] = rho * vy
        U[:, 3] = rho * vz
        U[:, 4] = 0.5 * rho * (vx ** 2 + vy ** 2 + vz ** 2) + p / (g - 1.0) + 0.5 * (bx ** 2 + by ** 2)
        U[:, 5] = bx
        U[:, 6] = by
        return U
    if c["ic"] == "shock":
        # Brio-Wu states, densities and pressures within 5 per cent of the usual ones
        f = 1.0 + 0.05 * rng.uniform(-1, 1, 4)
        left = X < 0.5 * box[0]
        rho = np.where(left, f[0], 0.125 * f[1]) * (1.0 + 1.0e-3 * rng.uniform(-1, 1, full))
        p = np.where(left, f[2], 0.1 * f[3])
        by = np.where(left, 1.0, -1.0)
        U[:, 0] = rho
        U[:, 4] = p / (g - 1.0) + 0.5 * (0.75 ** 2 + by ** 2)
        U[:, 5] = 0.75
        U[:, 6] = by
        return U
    if c["ic"] == "blast":
        # a hot sphere near the centre of a quiet, slightly noisy medium
        rho = 1.0 + 1.0e-3 * rng.uniform(-1, 1, full)
        cen = [b * (0.5 + 0.1 * q) for b, q in zip(box, rng.uniform(-1, 1, 3))]
        r0 = 0.12 * min(box)
        r2 = (X - cen[0]) ** 2 + (Y - cen[1]) ** 2 + (Z - cen[2]) ** 2
        p = np.where(r2 <= r0 * r0, 100.0, 1.0e-2)
    else:
        # ambient medium of 1 cm^-3 near 2e4 K; the remnant's is clumpy and
        # holds a hot sphere, the winds' carries 5 per cent noise
        if c["ic"] == "clumps":
            G = np.zeros(full)
            for _ in range(8):
                k = rng.normal(size=3)
                k *= 2.0 * math.pi * rng.uniform(1.5, 4.0) / np.linalg.norm(k) / max(box)
                G = G + np.cos(k[0] * X + (k[1] * Y + (k[2] * Z + rng.uniform(0.0, 2.0 * math.pi))))
            rho = np.exp(0.25 * G)
        else:
            rho = 1.0 + 0.05 * rng.uniform(-1, 1, full)
        p_sc = d_sc * v_sc ** 2
        p = rho * d_sc / (MU0 * AMU) * KB * 2.0e4 / p_sc
        if c["ic"] == "clumps":
            cen = [b * (0.5 + 0.03 * q) for b, q in zip(box, rng.uniform(-1, 1, 3))]
            r0 = 0.1 * min(box)
            r2 = (X - cen[0]) ** 2 + (Y - cen[1]) ** 2 + (Z - cen[2]) ** 2
            p = np.where(r2 <= r0 * r0, 3.0e3 * p, p)
    U[:, 0] = rho
    U[:, 4] = p / (g - 1.0)
    return U


# ---------------------------------------------------------------------------
# The framework's side
# ---------------------------------------------------------------------------
_BC = {"f": "free", "r": "reflective", "p": "periodic"}
_FORM = {"plain": 0, "fused32": 1, "fused64": 2}


def prepare(case, seed):
    from walicxe3d_amd import hip
    from walicxe3d_amd import workloads as W
    mhd = case["ic"] in ("ot", "shock")
    l_sc, d_sc, v_sc = _units(case)
    w = W.Workload(name="case", mhd=mhd, solver=case["solver"], limiter=case["limiter"], gamma_expr="",
                   gamma=_gamma(case), cfl=0.4, visc_eta=case["visc"], eight_wave=mhd,
                   bc=tuple(_BC[b] for b in case["bc"]), nroot=(case["nx"], case["ny"], case["nz"]),
                   maxlev=_top(case), phys=_phys(case), ic="ambient", seed=0, nsteps=0,
                   cooling=bool(case.get("cooling")), mu0=MU0, mui=MUI, l_sc=l_sc, d_sc=d_sc, v_sc=v_sc)
    mesh = _mesh(case)
    table, winds = _table(), _winds(case)
    # the problem's cooling curve and sources in place of the workload's own
    own = W.cooling_table, W.wind_params
    W.cooling_table, W.wind_params = (lambda *a, **k: table), (lambda *a, **k: winds)
    try:
        sim = hip.Walicxe3D(w, form=_FORM[case["form"]], bids=_block_ids(case, mesh))
    finally:
        W.cooling_table, W.wind_params = own
    sim.upload(_initial(case, mesh, seed))
    state = {"sim": sim, "steps": case["steps"], "regrid": None}
    if case.get("regrid"):
        state["regrid"] = (_block_ids(case, mesh), _block_ids(case, _mesh(case, 1.15)))
    return state


def run(state):
    sim, n = state["sim"], state["steps"]
    if state["regrid"] is None:
        sim.run(n)
        return {"U": sim.download(prim=False), "time": sim.time.value}
    small, large = state["regrid"]
    sim.record_ghosts()
    sim.run(1)
    flags, grad = sim.markByPhysical()
    sim.remesh(large)
    sim.run(n // 2)
    sim.remesh(small)
    sim.run(n - n // 2)
    return {"U": sim.download(prim=False), "time": sim.time.value, "flags": flags, "grad": grad}


def work(case):
    """State read and written once per step, and downloaded once; the
    operations of the reconstruction, the Riemann solver (three faces per
    cell and stage), the primitives, the update and the timestep."""
    zones = len(_mesh(case)) * NC ** 3
    nv = 8 if case["ic"] in ("ot", "shock") else 5
    steps = case["steps"] + (1 if case.get("regrid") else 0)
    face = {"hll": 90, "hllc": 100, "hlle": 180, "hlld": 300}[case["solver"]]
    cell = 2 * 3 * face + 3 * 12 * nv + 2 * (25 + 10 * nv) + 30 + (9 * nv if case["visc"] else 0)
    cell += 120 if case.get("cooling") else 0
    return {"bytes": zones * nv * 8 * (2 * steps + 1), "flops": zones * steps * cell}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch.  Arrays are [variable][block][z][y][x].
# ---------------------------------------------------------------------------
class _Exact:
    def __init__(self, c, mesh):
        self.c, self.mhd = c, c["ic"] in ("ot", "shock")
        self.nv = 8 if self.mhd else 5
        self.gamma = _gamma(c)
        self.cv = 1.0 / (self.gamma - 1.0)
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        l_sc, d_sc, v_sc = _units(c)
        self.l_sc, self.d_sc, self.v_sc, self.p_sc, self.t_sc = l_sc, d_sc, v_sc, d_sc * v_sc ** 2, l_sc / v_sc
        t, lam = _table()
        self.tabT, self.tabL = self.put(t), self.put(lam)
        self.it, self.time = 0, 0.0
        self.set_mesh(mesh)

    def put(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)

    def set_mesh(self, mesh):
        c, self.mesh = self.c, mesh
        at = {m: n for n, m in enumerate(mesh)}
        self.dx = self.put(np.array([_dx(c, m[0]) for m in mesh]).T)[:, :, None, None, None]
        r = np.arange(NC)
        A2, A1 = np.meshgrid(r, r, indexing="ij")
        A1, A2 = A1.ravel(), A2.ravel()
        one = {k: [] for k in ("dst", "src", "layer")}
        neg = {d: [] for d in range(3)}
        eight = {k: [] for k in ("dst", "src", "layer")}

        def cell(b, q):                       # flat interior index of cell q (0-based x, y, z)
            return ((b * NC + q[2]) * NC + q[1]) * NC + q[0]

        def ghost(b, q):                      # flat index with ghosts
            return ((b * NB + q[2] + 2) * NB + q[1] + 2) * NB + q[0] + 2

        def spread(d, n, a1, a2):             # normal and transverse coordinates to x, y, z
            t1, t2 = [a for a in range(3) if a != d]
            q = [None] * 3
            q[d], q[t1], q[t2] = np.broadcast_to(n, a1.shape), a1, a2
            return q

        for b, m in enumerate(mesh):
            l, p = m[0], m[1:]
            n = _dims(c, l)
            for f in range(6):
                d, low = f >> 1, (f & 1) == 0
                t1, t2 = [a for a in range(3) if a != d]
                nb = list(p)
                nb[d] += -1 if low else 1
                edge = not 0 <= nb[d] < n[d]
                kind = c["bc"][f] if edge else ""
                if kind == "p":
                    nb[d] %= n[d]
                for g in (1, 2):
                    dst = ghost(b, spread(d, -g if low else NC - 1 + g, A1, A2))
                    if kind in ("f", "r"):
                        # open: the edge cell at low faces, mirrored at high ones; wall: mirrored, normal momentum
                        # turned
                        k = (0 if low else NC - g) if kind == "f" else (g - 1 if low else NC - g)
                        src = cell(b, spread(d, k, A1, A2))
                        if kind == "r":
                            neg[d].append(dst)
                    elif (l, *nb) in at:
                        src = cell(at[(l, *nb)], spread(d, NC - g if low else g - 1, A1, A2))
                    elif (l - 1, nb[0] >> 1, nb[1] >> 1, nb[2] >> 1) in at:
                        o = at[(l - 1, nb[0] >> 1, nb[1] >> 1, nb[2] >> 1)]
                        src = cell(o, spread(d, NC - 1 if low else 0, (A1 >> 1) + (p[t1] & 1) * 8,
                                             (A2 >> 1) + (p[t2] & 1) * 8))
                    else:
                        kids = np.empty((2, 2), dtype=np.int64)
                        for s1 in (0, 1):
                            for s2 in (0, 1):
                                q = [2 * v for v in nb]
                                q[d] += 1 if low else 0
                                q[t1] += s1
                                q[t2] += s2
                                kids[s1, s2] = at[(l + 1, *q)]
                        o = kids[A1 >> 3, A2 >> 3]
                        k = NC - 2 * g if low else 2 * g - 2
                        src = np.stack([cell(o, spread(d, k + i, 2 * (A1 & 7) + j, 2 * (A2 & 7) + h))
                                        for i in (0, 1) for j in (0, 1) for h in (0, 1)])
                        eight["dst"].append(dst)
                        eight["src"].append(src)
                        eight["layer"].append(g)
                        continue
                    one["dst"].append(dst)
                    one["src"].append(src)
                    one["layer"].append(g)

        def index(v):
            return torch.as_tensor(np.concatenate(v, axis=-1), device=self.dev) if v else None

        self.copy = {g: (index([x for x, y in zip(one["dst"], one["layer"]) if y == g]),
                         index([x for x, y in zip(one["src"], one["layer"]) if y == g])) for g in (1, 2)}
        self.mean = {g: (index([x for x, y in zip(eight["dst"], eight["layer"]) if y == g]),
                         index([x for x, y in zip(eight["src"], eight["layer"]) if y == g])) for g in (1, 2)}
        self.turn = {d: index(v) for d, v in neg.items()}
        self.set_winds()

    def set_winds(self):
        """State and place (with ghosts) of the cells that a source covers."""
        self.wind_at = None
        winds = _winds(self.c)
        if not winds:
            return
        org = torch.tensor([m[1:] for m in self.mesh], dtype=torch.float64, device=self.dev) * NC
        q = torch.arange(-2, NC + 2, dtype=torch.float64, device=self.dev) + 0.5
        dx = self.dx.reshape(3, -1)
        ax = [(org[:, d, None] + q[None, :]) * dx[d][:, None] * self.l_sc for d in range(3)]
        X, Y, Z = ax[0][:, None, None, :], ax[1][:, None, :, None], ax[2][:, :, None, None]
        st = torch.zeros((5, len(self.mesh), NB, NB, NB), dtype=torch.float64, device=self.dev)
        hit = torch.zeros((len(self.mesh), NB, NB, NB), dtype=torch.bool, device=self.dev)
        for x, y, z, rad, mdot, v, temp, mu in winds:
            dist = torch.sqrt((X - x) ** 2 + (Y - y) ** 2 + (Z - z) ** 2)
            m = dist < rad
            rho = mdot / v / dist / dist / (4.0 * PI_REF)
            prim = [rho / self.d_sc, v * (X - x) / dist / self.v_sc, v * (Y - y) / dist / self.v_sc,
                    v * (Z - z) / dist / self.v_sc, rho / (mu * AMU) * KB * temp / self.p_sc]
            u = self.conserved(torch.stack([a.expand_as(dist) for a in prim]))
            st = torch.where(m[None], u, st)
            hit |= m
        self.wind_at = hit.reshape(-1).nonzero()[:, 0]
        self.wind_u = st.reshape(5, -1)[:, self.wind_at]

    # -- states -----------------------------------------------------------
    def prims(self, u):
        v = u[1:4] / u[0]
        p = u[4] - 0.5 * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / u[0]
        if self.mhd:
            p = p - 0.5 * (u[5] ** 2 + u[6] ** 2 + u[7] ** 2)
        p = torch.clamp(p / self.cv, min=1.0e-30)
        return torch.cat([torch.clamp(u[0], min=1.0e-40)[None], v, p[None], u[5:]])

    def conserved(self, w):
        e = 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) + self.cv * w[4]
        if self.mhd:
            e = e + 0.5 * (w[5] ** 2 + w[6] ** 2 + w[7] ** 2)
        return torch.cat([w[0:1], w[0] * w[1:4], e[None], w[5:]])

    def ghosts(self, U, depth):
        """U with its face ghosts; edge and corner ghosts hold ones."""
        nv, nb = U.shape[:2]
        G = torch.ones((nv, nb, NB, NB, NB), dtype=torch.float64, device=self.dev)
        G[:, :, 2:-2, 2:-2, 2:-2] = U
        flat, src = G.view(nv, -1), U.reshape(nv, -1)
        for g in range(1, depth + 1):
            dst, at = self.copy[g]
            flat[:, dst] = src[:, at]
            dst, at = self.mean[g]
            if dst is not None:
                flat[:, dst] = sum(src[:, a] for a in at) / 8.0
        for d, dst in self.turn.items():
            if dst is not None:
                flat[1 + d, dst] *= -1.0
        if self.wind_at is not None:
            flat[:, self.wind_at] = self.wind_u
        return G

    # -- fluxes -----------------------------------------------------------
    def flux_of(self, w):
        v2 = w[1] ** 2 + w[2] ** 2 + w[3] ** 2
        e = 0.5 * w[0] * v2 + (self.cv + 1.0) * w[4]
        if not self.mhd:
            return torch.stack([w[0] * w[1], w[0] * w[1] ** 2 + w[4], w[0] * w[1] * w[2], w[0] * w[1] * w[3],
                                w[1] * e])
        b2 = w[5] ** 2 + w[6] ** 2 + w[7] ** 2
        vb = w[1] * w[5] + w[2] * w[6] + w[3] * w[7]
        return torch.stack([w[0] * w[1], w[0] * w[1] ** 2 + w[4] + 0.5 * b2 - w[5] ** 2,
                            w[0] * w[1] * w[2] - w[5] * w[6], w[0] * w[1] * w[3] - w[5] * w[7],
                            w[1] * (e + b2) - w[5] * vb, torch.zeros_like(vb), w[1] * w[6] - w[2] * w[5],
                            w[1] * w[7] - w[3] * w[5]])

    def fast(self, w, axis=1):
        """Fast speed along an axis (sound speed in hydro)."""
        if not self.mhd:
            return torch.sqrt(self.gamma * w[4] / w[0])
        a = self.gamma * w[4] + w[5] ** 2 + w[6] ** 2 + w[7] ** 2
        root = torch.sqrt(torch.clamp(a * a - 4.0 * self.gamma * w[4] * w[4 + axis] ** 2, min=0.0))
        return torch.sqrt(0.5 * (a + root) / w[0])

    def riemann(self, L, R):
        cl, cr = self.fast(L), self.fast(R)
        sl, sr = torch.minimum(L[1] - cl, R[1] - cr), torch.maximum(L[1] + cl, R[1] + cr)
        FL, FR = self.flux_of(L), self.flux_of(R)
        s = self.c["solver"]
        if s in ("hll", "hlle"):
            mid = (sr * FL - sl * FR + sl * sr * (self.conserved(R) - self.conserved(L))) / (sr - sl)
        elif s == "hllc":
            mid = self.contact(L, R, FL, FR, sl, sr)
        else:
            mid = self.hlld(L, R, FL, FR, sl, sr)
        return torch.where(sl > 0, FL, torch.where(sr < 0, FR, mid))

    def contact(self, L, R, FL, FR, sl, sr):
        ml, mr = L[0] * (sl - L[1]), R[0] * (sr - R[1])
        sm = (R[4] - L[4] + L[1] * ml - R[1] * mr) / (ml - mr)

        def side(w, F, s, m):
            u = self.conserved(w)
            rho = m / (s - sm)
            e = rho * (u[4] / w[0] + (sm - w[1]) * (sm + w[4] / m))
            return F + s * (torch.stack([rho, rho * sm, rho * w[2], rho * w[3], e]) - u)

        return torch.where(sm >= 0, side(L, FL, sl, ml), side(R, FR, sr, mr))

    def hlld(self, L, R, FL, FR, sl, sr):
        """Miyoshi & Kusano (2005), with the mean normal field in the fan."""
        bx = 0.5 * (L[5] + R[5])
        sign = torch.where(bx >= 0, 1.0, -1.0).to(bx)
        ml, mr = L[0] * (sl - L[1]), R[0] * (sr - R[1])
        ptl = L[4] + 0.5 * (bx ** 2 + L[6] ** 2 + L[7] ** 2)
        ptr = R[4] + 0.5 * (bx ** 2 + R[6] ** 2 + R[7] ** 2)
        sm = (mr * R[1] - ml * L[1] - ptr + ptl) / (mr - ml)
        pst = (mr * ptl - ml * ptr + ml * mr * (R[1] - L[1])) / (mr - ml)

        def star(w, s, m, pt):
            rho = m / (s - sm)
            den = m * (s - sm) - bx ** 2
            ok = den != 0
            den = torch.where(ok, den, torch.ones_like(den))
            k = bx * (sm - w[1]) / den
            h = (m * (s - w[1]) - bx ** 2) / den
            zero = torch.zeros_like(den)
            v, q = torch.where(ok, w[2] - k * w[6], w[2]), torch.where(ok, w[3] - k * w[7], w[3])
            by, bz = torch.where(ok, h * w[6], zero), torch.where(ok, h * w[7], zero)
            e = 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) + self.cv * w[4] + pt - w[4]
            vb, vbs = w[1] * bx + w[2] * w[6] + w[3] * w[7], sm * bx + v * by + q * bz
            e = ((s - w[1]) * e - pt * w[1] + pst * sm + bx * (vb - vbs)) / (s - sm)
            return rho, v, q, by, bz, e, vbs

        def fan(rho, v, q, by, bz, e, vb):
            return torch.stack([rho * sm, rho * sm ** 2 + pst - bx ** 2, rho * sm * v - bx * by,
                                rho * sm * q - bx * bz, sm * (e + pst) - bx * vb, torch.zeros_like(sm),
                                by * sm - bx * v, bz * sm - bx * q])

        rl, vl, wl, byl, bzl, el, vbl = star(L, sl, ml, ptl)
        rr, vr, wr, byr, bzr, er, vbr = star(R, sr, mr, ptr)
        ql, qr = torch.sqrt(rl), torch.sqrt(rr)
        sal, sar = sm - bx.abs() / ql, sm + bx.abs() / qr
        t = ql + qr
        v = (ql * vl + qr * vr + (byr - byl) * sign) / t
        q = (ql * wl + qr * wr + (bzr - bzl) * sign) / t
        by = (ql * byr + qr * byl + ql * qr * (vr - vl) * sign) / t
        bz = (ql * bzr + qr * bzl + ql * qr * (wr - wl) * sign) / t
        vb = sm * bx + v * by + q * bz
        out = torch.where(sm >= 0, fan(rl, v, q, by, bz, el - ql * (vbl - vb) * sign, vb),
                          fan(rr, v, q, by, bz, er + qr * (vbr - vb) * sign, vb))
        out = torch.where(sar <= 0, fan(rr, vr, wr, byr, bzr, er, vbr), out)
        return torch.where(sal >= 0, fan(rl, vl, wl, byl, bzl, el, vbl), out)

    def average(self, a, b):
        lim = self.c["limiter"]
        s = torch.where(a >= 0, 1.0, -1.0).to(a)
        if lim == "minmod":
            return s * torch.clamp(torch.minimum(a.abs(), s * b), min=0.0)
        if lim == "vanleer":
            ab = a * b
            return torch.where(ab > 0, ab * (a + b) / torch.where(ab > 0, a * a + b * b, torch.ones_like(ab)),
                               torch.zeros_like(ab))
        if lim == "woodward":
            r = torch.minimum(torch.minimum(2.0 * a.abs(), 2.0 * s * b), s * 0.5 * (a + b))
            return s * torch.clamp(r, min=0.0)
        s = torch.where(b >= 0, 1.0, -1.0).to(a)           # superbee
        return s * torch.clamp(torch.maximum(torch.minimum(2.0 * b.abs(), s * a),
                                             torch.minimum(b.abs(), 2.0 * s * a)), min=0.0)

    def faces(self, P, d, order):
        """Fluxes at the 17 faces along axis d (0 x, 1 y, 2 z)."""
        dim = 4 - d
        sel = [slice(None), slice(None)] + [slice(2, -2)] * 3
        turn = list(range(self.nv))
        turn[1], turn[1 + d] = turn[1 + d], turn[1]
        if self.mhd:
            turn[5], turn[5 + d] = turn[5 + d], turn[5]

        def at(o):
            sel[dim] = slice(1 + o, 18 + o)
            return P[tuple(sel)][turn]

        L, R = at(0), at(1)
        if order == 2:
            dl, dm, dr = L - at(-1), R - L, at(2) - R
            L, R = L + 0.5 * self.average(dl, dm), R - 0.5 * self.average(dm, dr)
        return self.riemann(L, R)[turn]

    def update(self, U, P, dt, order):
        out = torch.empty_like(U)
        step = 1024
        for b in range(0, U.shape[1], step):
            e = min(U.shape[1], b + step)
            p, dx, new = P[:, b:e], self.dx[:, b:e], U[:, b:e].clone()
            for d in range(3):
                F = self.faces(p, d, order)
                dim = 4 - d
                new += dt / dx[d] * (F.narrow(dim, 0, NC) - F.narrow(dim, 1, NC))
            if self.mhd:
                w = p[:, :, 2:-2, 2:-2, 2:-2]
                div = ((p[5, :, 2:-2, 2:-2, 3:-1] - p[5, :, 2:-2, 2:-2, 1:-3]) / (2.0 * dx[0]) +
                       (p[6, :, 2:-2, 3:-1, 2:-2] - p[6, :, 2:-2, 1:-3, 2:-2]) / (2.0 * dx[1]) +
                       (p[7, :, 3:-1, 2:-2, 2:-2] - p[7, :, 1:-3, 2:-2, 2:-2]) / (2.0 * dx[2]))
                new[1:4] -= dt * div * w[5:8]
                new[4] -= dt * div * (w[1] * w[5] + w[2] * w[6] + w[3] * w[7])
                new[5:8] -= dt * div * w[1:4]
            out[:, b:e] = new
        return out

    def cool(self, U, dt):
        w = self.prims(U)
        temp = w[4] / w[0] * (MU0 * AMU * self.p_sc / self.d_sc / KB)
        logt = torch.log10(temp)
        n = len(self.tabT)
        hi = torch.clamp(torch.searchsorted(self.tabT, logt.reshape(-1), right=True).reshape(logt.shape), 1, n - 1)
        t0, t1, c0, c1 = self.tabT[hi - 1], self.tabT[hi], self.tabL[hi - 1], self.tabL[hi]
        lam = torch.pow(10.0, (c1 - c0) / (t1 - t0) * (logt - t0) + c0)
        lam = torch.where(logt >= self.tabT[-1], torch.pow(10.0, self.tabL[-1] + 0.5 * (logt - self.tabT[-1])), lam)
        eth = self.cv * w[4]
        num = w[0] * self.d_sc / (MUI * AMU)
        fac = torch.exp(-lam * num ** 2 / (eth * self.p_sc) * (dt * self.t_sc))
        fac = torch.clamp(fac, min=0.5)
        fac = torch.where(temp * fac < 10.0, 10.0 / temp, fac)
        e = 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) + eth * fac
        out = U.clone()
        out[4] = torch.where(logt >= self.tabT[0], e, U[4])
        return out

    def timestep(self, U):
        w = self.prims(U)
        return min(float((self.dx[d] / (w[1 + d].abs() + self.fast(w, 1 + d))).min()) for d in range(3)) * 0.4

    def step(self, U):
        self.it += 1
        dt = self.timestep(U)
        if self.it <= 10:
            dt *= 2.0 ** -(11 - self.it)
        before = self.prims(U)
        G = self.ghosts(U, 1)
        P = self.prims(G)
        P[:, :, 2:-2, 2:-2, 2:-2] = before      # the predictor's interior is that before the sources are imposed
        U = G[:, :, 2:-2, 2:-2, 2:-2].clone()
        half = self.update(U, P, 0.5 * dt, 1)
        G = self.ghosts(half, 2)
        new = self.update(U, self.prims(G), dt, 2)
        if self.c["visc"]:
            G[:, :, 2:-2, 2:-2, 2:-2] = new
            m = slice(2, -2)
            lap = (G[:, :, m, m, 3:-1] + G[:, :, m, m, 1:-3] + G[:, :, m, 3:-1, m] + G[:, :, m, 1:-3, m] +
                   G[:, :, 3:-1, m, m] + G[:, :, 1:-3, m, m] - 6.0 * new)
            new = new + self.c["visc"] * lap
        if self.c.get("cooling"):
            new = self.cool(new, dt)
        self.time += dt
        return new

    # -- mesh changes -----------------------------------------------------
    def gradients(self, before, U):
        """Largest relative gradient of pressure and density per block, with
        the ghost layer of the state before the step."""
        P = self.prims(self.ghosts(before, 1))
        P[:, :, 2:-2, 2:-2, 2:-2] = self.prims(U)
        m, out = slice(2, -2), None
        for v in (0, 4):
            q = P[v]
            for hi, lo in ((q[:, m, m, 3:-1], q[:, m, m, 1:-3]), (q[:, m, 3:-1, m], q[:, m, 1:-3, m]),
                           (q[:, 3:-1, m, m], q[:, 1:-3, m, m])):
                g = ((hi - lo).abs() / q[:, m, m, m] / (2.0 * self.dx[0])).amax(dim=(1, 2, 3))
                out = g if out is None else torch.maximum(out, g)
        return out

    def remesh(self, U, mesh):
        old = {m: n for n, m in enumerate(self.mesh)}
        new = torch.empty((self.nv, len(mesh), NC, NC, NC), dtype=torch.float64, device=self.dev)
        r = torch.arange(NC, device=self.dev)
        for n, (l, x, y, z) in enumerate(mesh):
            if (l, x, y, z) in old:
                new[:, n] = U[:, old[(l, x, y, z)]]
                continue
            up = next((k for k in range(1, l) if (l - k, x >> k, y >> k, z >> k) in old), None)
            if up is not None:
                src = U[:, old[(l - up, x >> up, y >> up, z >> up)]]
                at = [((q * NC + r) >> up) - (q >> up) * NC for q in (x, y, z)]
                new[:, n] = src[:, at[2]][:, :, at[1]][:, :, :, at[0]]
                continue
            for k in range(8):
                i, j, h = k & 1, (k >> 1) & 1, k >> 2
                kid = U[:, old[(l + 1, 2 * x + i, 2 * y + j, 2 * z + h)]]
                new[:, n, 8 * h:8 * h + 8, 8 * j:8 * j + 8, 8 * i:8 * i + 8] = kid.reshape(
                    -1, 8, 2, 8, 2, 8, 2).sum(dim=(2, 4, 6)) / 8.0
        self.set_mesh(mesh)
        return new


def exact(case, seed):
    mesh = _mesh(case)
    s = _Exact(case, mesh)
    U = s.put(np.moveaxis(_initial(case, mesh, seed), 1, 0))
    n = case["steps"]
    if not case.get("regrid"):
        for _ in range(n):
            U = s.step(U)
        return {"U": U.transpose(0, 1).contiguous(), "time": s.time}
    before, U = U, s.step(U)
    grad = s.gradients(before, U)
    U = s.remesh(U, _mesh(case, 1.15))
    for _ in range(n // 2):
        U = s.step(U)
    U = s.remesh(U, mesh)
    for _ in range(n - n // 2):
        U = s.step(U)
    return {"U": U.transpose(0, 1).contiguous(), "time": s.time, "flags": None, "grad": grad}
