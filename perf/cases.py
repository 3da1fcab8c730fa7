"""Performance cases: the work a user of spammm_amd has it do, over the range of sizes in use.

Single stages through the device layer (force-field grids, relaxed scans, the FDBM and Ewald field
producers) and whole calls (a differentiable image with its gradients, gridless and on a grid, a
batch of molecules).  Sizes follow spammm_amd.workloads, the tests and the benchmark.  ``exact``
recomputes a case in float64 with plain torch and numpy.

A relaxed scan stops at the first FIRE step with |F|^2 below f2conv, so at the loose default
(1e-8) a last-bit change of the grid moves single probe positions by up to |F|/k.  The scan cases
therefore relax on a grid made here, and the whole calls relax to |F| < 1e-6 (f2conv 1e-12) at
imaging heights, where the probe's equilibrium is unique.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from spammm_amd import _lib, batch, df as DF, device as D, diff, ewald, fdbm, workloads as W
from spammm_amd.params import ELEMENTS_BENCH, mix_R0E0, mix_lj, stiffness_Nm_to_eVA2

DEV = "cuda:0"
COULOMB = 14.3996448915
R2SAFE = 1e-4
EV_A2_TO_N_M = 16.02176634
TIGHT = dict(max_iter=1000, f2conv=1e-12)
# (charges, z offsets) of the tip: one charge on the probe, or AFMulator's default pair behind it
TIPS = {"point": ([W.PROBE_Q, 0, 0, 0], [0, 0, 0, 0]), "pair": ([0, -0.1, 0.1, 0], [0, 1.8, 3.6, 0]),
        "none": ([0, 0, 0, 0], [0, 0, 0, 0])}


# ── the cases ─────────────────────────────────────────────────────────────────────────

def _grid(name=None, **kw):
    c = dict(kind="grid", model="lj", atoms=60, cells=0, nx=200, ny=200, nz=200, step=0.1, npbc=1, tip="point",
             base=False, z0=-6.0)
    if name:
        c["name"] = name
    c.update(kw)
    return c


def listed():
    return [
        # the small coarse grid of a quick look or a test: latency and launches
        _grid("grid_small", atoms=18, nx=48, ny=40, nz=40, step=0.25, z0=-3.0),
        # one molecule of ordinary size with its periodic images, LJ + probe charge
        _grid("grid_flake", atoms=200, nx=300, ny=300, nz=240, z0=-8.0),
        # a free molecule under AFMulator's default tip (two charges behind the probe), Morse, odd sizes
        _grid("grid_morse", model="morse", atoms=97, nx=251, ny=233, nz=171, npbc=0, tip="pair", z0=-5.0),
        # the raw field of a substrate slab, done once per surface, on a fine grid
        _grid("grid_slab", cells=8, atoms=0, nx=320, ny=320, nz=96, step=0.05, z0=1.5),
        # one placement of a molecule over that surface's field: the inner loop of a placement search
        _grid("grid_placement", atoms=60, nx=480, ny=480, nz=149, step=0.05, base=True, z0=0.3),
        # a relaxed scan with its frequency shift on a grid at hand: what every image costs after its grid
        dict(name="scan_flake", kind="scan", atoms=200, nx=300, ny=300, nz=240, step=0.1, px=256, py=256, pz=60,
             strokes=False),
        # the relaxed strokes of a small FDBM image
        dict(name="scan_strokes", kind="scan", atoms=38, nx=200, ny=160, nz=200, step=0.1, px=100, py=80, pz=31,
             strokes=True),
        # the FDBM force field from densities: FFT overlap and electrostatics, dispersion, force grid
        dict(name="fdbm_fields", kind="fdbm", nx=200, ny=160, nz=128, step=0.1, atoms=38),
        # the periodic Coulomb field of an ionic slab
        dict(name="ewald_slab", kind="ewald", cells=8, nx=902, ny=902, nz=120, step=0.05, n_harm=40, tip="point"),
        # gridless Morse image and the gradients of its loss: a step of a fit of atom parameters
        dict(name="direct_fit", kind="direct", atoms=128, px=64, py=64, pz=60),
        # grid image and the gradients of its loss: a step of a structure fit
        dict(name="image_fit", kind="fit", atoms=200, nx=300, ny=300, nz=240, step=0.1, px=128, py=128, pz=40,
             params=False),
        # many molecules in one launch: images of a library of structures
        dict(name="batch_images", kind="batch", mols=24, max_atoms=150, px=128, pz=28),
    ]


def _lu(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _side(atoms):
    """Edge (A) of a cell that holds a flat flake of `atoms` atoms with a few A around it."""
    return 2.0 * math.sqrt(atoms / (0.3 * math.pi)) + 5.0


def draw(rng):
    kind = rng.choice(["grid"] * 5 + ["scan", "scan", "fdbm", "ewald", "direct", "fit", "batch"])
    if kind == "grid":
        step = rng.choice([0.05, 0.08, 0.1, 0.1, 0.1, 0.125, 0.15, 0.2, 0.25])
        if rng.random() < 0.2:
            n = _lu(rng, 60, 300)
            return _grid(cells=rng.randint(2, 6), atoms=0, nx=n, ny=n + rng.randint(-7, 7), nz=_lu(rng, 12, 90),
                         step=step, z0=1.5)
        atoms = _lu(rng, 8, 200)
        c = _grid(atoms=atoms, model=rng.choice(["lj", "lj", "morse"]), npbc=rng.choice([0, 1, 1]),
                  tip=rng.choice(["point", "point", "pair", "none"]), base=rng.random() < 0.25, step=step)
        ext = _side(atoms)
        c["nx"] = int(ext * rng.uniform(0.9, 1.2) / step) + rng.randint(0, 3)
        c["ny"] = int(ext * rng.uniform(0.9, 1.2) / step) + rng.randint(0, 3)
        c["nz"] = _lu(rng, 9, int(24 / step))
        c["z0"] = round(rng.uniform(-8.0, 3.0), 3)
        most = 200 * 9 * 300 * 300 * 240
        while c["nx"] * c["ny"] * c["nz"] > min(9e7, most / (atoms * (2 * c["npbc"] + 1) ** 2)):
            c["nz"] = max(9, c["nz"] // 2)
            c["nx"], c["ny"] = int(c["nx"] * 0.8), int(c["ny"] * 0.8)
        return c
    if kind == "scan":
        n = _lu(rng, 90, 300)
        px = _lu(rng, 11, 256)
        return dict(kind="scan", atoms=_lu(rng, 10, 200), nx=n, ny=n + rng.randint(-9, 9), nz=rng.randint(150, 240),
                    step=rng.choice([0.1, 0.1, 0.12]), px=px, py=max(5, px + rng.randint(-5, 5)),
                    pz=rng.randint(8, 60), strokes=rng.random() < 0.4)
    if kind == "fdbm":
        even = [n for n in range(48, 200, 2) if _smooth(n)]
        return dict(kind="fdbm", nx=rng.choice(even), ny=rng.choice(even), nz=rng.choice(even),
                    step=rng.choice([0.1, 0.15, 0.2]), atoms=_lu(rng, 8, 60))
    if kind == "ewald":
        n = _lu(rng, 60, 700)
        return dict(kind="ewald", cells=rng.randint(1, 8), nx=n, ny=n + rng.randint(-9, 9), nz=_lu(rng, 17, 120),
                    step=rng.choice([0.05, 0.1, 0.1, 0.2]), n_harm=rng.choice([4, 12, 24, 40]),
                    tip=rng.choice(["point", "pair"]))
    if kind == "direct":
        px = _lu(rng, 16, 64)
        return dict(kind="direct", atoms=_lu(rng, 8, 128), px=px, py=px + rng.randint(-3, 0), pz=rng.randint(20, 60))
    if kind == "fit":
        atoms = _lu(rng, 12, 160)
        n = int(max(12.0, _side(atoms)) / 0.1) + rng.randint(0, 9)
        return dict(kind="fit", atoms=atoms, nx=n, ny=n - rng.randint(0, 5), nz=rng.randint(200, 240), step=0.1,
                    px=_lu(rng, 32, 128), py=_lu(rng, 32, 128), pz=rng.randint(24, 40), params=rng.random() < 0.4)
    return dict(kind="batch", mols=_lu(rng, 2, 24), max_atoms=_lu(rng, 20, 150), px=_lu(rng, 32, 128),
                pz=rng.randint(20, 28))


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


# ── inputs (host, from the seed alone) ────────────────────────────────────────────────

def _rng(seed, salt):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, salt])


def _flake(atoms, rng):
    """(element names, (na,4) float32 x,y,z,q) of a flat flake, charges U(-0.3, 0.3) e, neutral."""
    en, pos = W.flake_geometry(atoms, rng)
    a = np.zeros((atoms, 4), np.float32)
    a[:, :3] = pos
    q = rng.uniform(-0.3, 0.3, atoms)
    a[:, 3] = q - q.mean()
    return en, a


def _spec(c, centred=True, z0=None):
    L = np.array([c["nx"], c["ny"], c["nz"]]) * c["step"]
    p0 = np.array([-L[0] / 2 if centred else 0.0, -L[1] / 2 if centred else 0.0, c["z0"] if z0 is None else z0])
    return D.axis_aligned_spec(p0, L, (c["nx"], c["ny"], c["nz"])), L.astype(np.float32)


def _slab(cells, rng):
    en, a = W.rocksalt_slab(cells)
    a = a + np.concatenate([rng.normal(0, 0.02, (len(en), 3)), np.zeros((len(en), 1))], 1).astype(np.float32)
    return en, a


def _grid_inputs(c, seed):
    """Host inputs of a grid case: atoms, pair parameters, lattice vectors, spec."""
    rng = _rng(seed, 1)
    if c["cells"]:
        en, a = _slab(c["cells"], rng)
        Lxy = c["cells"] * 5.64
        spec, _ = _spec(c, centred=False)
        lv = np.array([Lxy, Lxy], np.float32)
    else:
        en, a = _flake(c["atoms"], rng)
        if c["base"]:
            a[:, 2] += 3.0
        spec, L = _spec(c)
        lv = L[:2]
    if c["model"] == "lj":
        cp = mix_lj(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
    else:
        R0, E0 = mix_R0E0(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
        cp = np.stack([R0, E0, np.full(len(en), -1.8), np.zeros(len(en))], 1).astype(np.float32)
    cp = np.ascontiguousarray(cp, np.float32)
    lvA, lvB = np.array([lv[0], 0, 0], np.float32), np.array([0, lv[1], 0], np.float32)
    return a, cp, lvA, lvB, spec


def _base_field(c, seed):
    """A smooth substrate field (nz,ny,nx,4) float32: a few decaying in-plane harmonics."""
    g = torch.Generator(device="cpu").manual_seed(int(seed) + 77)
    r = torch.rand(8, 4, generator=g, dtype=torch.float32).to(DEV)
    x = torch.arange(c["nx"], device=DEV, dtype=torch.float32)[None, None, :] * c["step"]
    y = torch.arange(c["ny"], device=DEV, dtype=torch.float32)[None, :, None] * c["step"]
    z = torch.arange(c["nz"], device=DEV, dtype=torch.float32)[:, None, None] * c["step"]
    out = torch.empty((c["nz"], c["ny"], c["nx"], 4), device=DEV)
    for k in range(4):
        ph = 1.1141 * (x + (k % 2) * y) + 6.28 * r[k, 0]
        out[..., k] = 0.05 * (0.3 + r[k, 1]) * torch.exp(-1.1 * z) * torch.cos(ph) * torch.cos(1.1141 * y + r[k, 2])
    return out


def _tip(dz=-0.1, bond=4.0):
    kl, kr = stiffness_Nm_to_eVA2(0.25), stiffness_Nm_to_eVA2(20.0)
    return D.Tip(stiffness=np.array([-kl, -kl, -kl, -kr], np.float32),
                 dpos0=np.array([0, 0, -bond, bond], np.float32), tipC=np.array([0, 0, 1, dz], np.float32))


def _raster(L, px, py, z):
    dx, dy = float(L[0]) / px, float(L[1]) / py
    return D.scan_points([-L[0] / 2 + dx / 2, -L[1] / 2 + dy / 2, z], [dx, 0, 0], [0, dy, 0], px, py)


def _target(a, px, py, pz, L, rng):
    """A measured-looking image (px, py, pz), Hz: a dip over each displaced atom, deeper when closer."""
    x = torch.as_tensor((np.arange(px) + 0.5) * L[0] / px - L[0] / 2, device=DEV, dtype=torch.float32)
    y = torch.as_tensor((np.arange(py) + 0.5) * L[1] / py - L[1] / 2, device=DEV, dtype=torch.float32)
    xy = torch.as_tensor(a[:, :2] + rng.normal(0, 0.1, (len(a), 2)), device=DEV, dtype=torch.float32)
    gx = torch.exp(-(x[:, None] - xy[None, :, 0]) ** 2 / 2.0)
    gy = torch.exp(-(y[:, None] - xy[None, :, 1]) ** 2 / 2.0)
    ramp = torch.linspace(0.02, 1.0, pz, device=DEV) ** 2
    return ((gx @ gy.T)[:, :, None] * (-0.8 * ramp)).contiguous()


def _fit_inputs(c, seed):
    rng = _rng(seed, 2)
    en, a = _flake(c["atoms"], rng)
    R0, E0 = mix_R0E0(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
    if c["kind"] == "fit":
        L = np.array([c["nx"], c["ny"], c["nz"]]) * c["step"]
    else:
        L = np.array([_side(c["atoms"])] * 2 + [0.0])
    top = 7.7 + 0.1 * (c["pz"] - 1)
    return a, np.asarray(R0, np.float32), np.asarray(E0, np.float32), L, top, rng


def _scan_grid(c, seed):
    """A force-field grid of a flake made with plain torch (nearest image in x, y), (nz,ny,nx,4)."""
    en, a = _flake(c["atoms"], _rng(seed, 3))
    cp = mix_lj(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
    spec, L = _spec(c, z0=-8.0)
    ax = [torch.arange(n, device=DEV, dtype=torch.float32) * c["step"] + float(o) for n, o in zip(spec.n, spec.p0)]
    fr = [torch.zeros(c["nz"], c["ny"], c["nx"], device=DEV) for _ in range(4)]
    for (x, y, z, q), (c6, c12) in zip(a.tolist(), np.asarray(cp).tolist()):
        dx = ax[0] - x
        dy = ax[1] - y
        dx = (dx - L[0] * torch.round(dx / L[0]))[None, None, :]
        dy = (dy - L[1] * torch.round(dy / L[1]))[None, :, None]
        dz = (ax[2] - z)[:, None, None]
        i2 = 1.0 / (dx * dx + (dy * dy + (dz * dz + R2SAFE)))
        i6 = i2 * i2 * i2
        ec = (COULOMB * W.PROBE_Q * q) * i2.sqrt()
        fr[3] += (c12 * i6 - c6) * i6 + ec
        f = ((12 * c12 * i6 - 6 * c6) * i6 + ec) * i2
        fr[0] += f * dx
        fr[1] += f * dy
        fr[2] += f * dz
    s = (100.0 / fr[3].abs()).clamp(max=1.0)
    return torch.stack([v * s for v in fr], -1).contiguous(), spec, L


def _batch_mols(c, seed):
    rng = _rng(seed, 4)
    out = []
    for k in range(c["mols"]):
        w = W.batch_molecule(k, base_seed=int(rng.integers(1 << 30)))
        if w.atoms.shape[0] > c["max_atoms"]:
            en, a = _flake(int(rng.integers(10, c["max_atoms"] + 1)), rng)
            w.enames, w.atoms = en, a
            w.cLJ = mix_lj(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
        step = float(w.L[0]) / c["px"]
        w.nxy, w.nz = (c["px"], c["px"]), c["pz"]
        w.scan_p0 = np.array([-w.L[0] / 2 + step / 2, -w.L[0] / 2 + step / 2, 7.9 + 0.1 * (c["pz"] - 1)], np.float32)
        w.scan_da, w.scan_db = np.array([step, 0, 0], np.float32), np.array([0, step, 0], np.float32)
        out.append(w)
    return out


def _fdbm_inputs(c, seed):
    rng = _rng(seed, 5)
    shape, st = (c["nx"], c["ny"], c["nz"]), c["step"]
    half = np.array(shape) * st / 2
    pos = np.concatenate([rng.uniform(-0.6, 0.6, (c["atoms"], 2)) * half[:2], rng.normal(0, 0.05, (c["atoms"], 1))], 1)
    Z = rng.choice([1, 6, 7, 8], c["atoms"]).astype(np.float64)
    q = rng.uniform(-0.3, 0.3, c["atoms"])
    q -= q.mean()

    def gauss(centres, sigma, weights, shp, org):
        ax = [torch.as_tensor(org[k] + st * np.arange(shp[k]), device=DEV, dtype=torch.float32) for k in range(3)]
        g = [torch.exp(-(ax[k][:, None] - torch.as_tensor(centres[:, k], device=DEV, dtype=torch.float32)) ** 2
                       / (2 * sigma * sigma)) for k in range(3)]
        w = torch.as_tensor(weights, device=DEV, dtype=torch.float32) / ((2 * math.pi) ** 1.5 * sigma ** 3)
        return torch.einsum("xa,ya,za->xyz", g[0], g[1], g[2] * w).contiguous()

    tip = np.zeros((1, 3))
    up = np.array([[0, 0, 0.2]])
    torg = -12 * st * np.ones(3)
    tot = gauss(tip, 0.6, [6.0], (24, 24, 24), torg)
    dlt = gauss(up, 0.5, [0.4], (24, 24, 24), torg) - gauss(-up, 0.5, [0.4], (24, 24, 24), torg)

    def rolled(t):
        p = torch.zeros(shape, device=DEV)
        p[:24, :24, :24] = t
        return torch.roll(p, (-12, -12, -12), (0, 1, 2)).contiguous()

    aw = np.zeros((c["atoms"], 4), np.float32)
    aw[:, :3] = pos
    aw[:, 3] = np.sqrt(30.0 * rng.uniform(2.0, 25.0, c["atoms"]))
    return dict(rho=gauss(pos, 0.55, Z, shape, -half), diff=(gauss(pos, 0.45, q, shape, -half)
                                                             - gauss(pos, 0.65, q, shape, -half)).contiguous(),
                tot=rolled(tot), dlt=rolled(dlt), atoms=torch.as_tensor(aw, device=DEV), origin=-half, step=st,
                shape=shape, A=18.0, beta=1.2)


def _ewald_inputs(c, seed):
    _, ions = W.rocksalt_slab(c["cells"])
    rng = _rng(seed, 6)
    ions = ions.copy()
    ions[:, 3] *= np.float32(rng.uniform(0.6, 1.1))
    Lxy = c["cells"] * 5.64
    spec = D.axis_aligned_spec([rng.uniform(-2, 2), rng.uniform(-2, 2), 1.5],
                               np.array([c["nx"], c["ny"], c["nz"]]) * c["step"], (c["nx"], c["ny"], c["nz"]))
    return ions, Lxy, spec


# ── prepare and run ───────────────────────────────────────────────────────────────────

def prepare(case, seed):
    c, k = case, case["kind"]
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=DEV)  # noqa: E731
    if k == "grid":
        a, cp, lvA, lvB, spec = _grid_inputs(c, seed)
        Qs, QZs = TIPS[c["tip"]]
        s = dict(args=(t(a), t(cp), _lib.PPM_MODEL_LJ if c["model"] == "lj" else _lib.PPM_MODEL_MORSE, spec, Qs, QZs,
                       (c["npbc"], c["npbc"]), lvA, lvB), cap=not c["cells"])
        s["base"] = _base_field(c, seed) if c["base"] else None
        s["out"] = torch.empty((c["nz"], c["ny"], c["nx"], 4), device=DEV)
    elif k == "scan":
        G, spec, L = _scan_grid(c, seed)
        pts = t(_raster(L, c["px"], c["py"], 12.0))
        op = DF.z_operator("giessibl", c["pz"], -0.1, DEV)
        n = c["px"] * c["py"]
        s = dict(grid=G, spec=spec, pts=pts, tip=_tip(), op=op, df=torch.empty((n, c["pz"]), device=DEV),
                 FEs=torch.empty((n, c["pz"], 4), device=DEV), PPs=torch.empty((n, c["pz"], 4), device=DEV))
    elif k == "fdbm":
        s = _fdbm_inputs(c, seed)
    elif k == "ewald":
        ions, Lxy, spec = _ewald_inputs(c, seed)
        s = dict(ew=ewald.SurfaceEwald(DEV).prepare_system(ions, [Lxy, 0], [0, Lxy], c["n_harm"]), spec=spec,
                 out=torch.empty((c["nz"], c["ny"], c["nx"], 4), device=DEV))
    elif k in ("fit", "direct"):
        a, R0, E0, L, top, rng = _fit_inputs(c, seed)
        Qs, QZs = (np.array(v, np.float32) for v in TIPS["point"])
        pts = t(_raster(L, c["px"], c["py"], top))
        common = dict(pts=pts, nxy=(c["px"], c["py"]), nz=c["pz"], tip=_tip(), Qs=Qs, QZs=QZs)
        if k == "fit":
            spec, _ = _spec(c, z0=-8.0)
            prob = diff.Problem(spec=spec, npbc=(1, 1), lvA=np.array([L[0], 0, 0], np.float32),
                                lvB=np.array([0, L[1], 0], np.float32), window_margin=(2.0, 1.0), **common)
        else:
            prob = diff.DirectProblem(**common)
        leaf = lambda v, g=True: t(v).requires_grad_(g)  # noqa: E731
        par = k == "direct" or c["params"]
        s = dict(leaves=(leaf(a[:, :3]), leaf(a[:, 3]), leaf(R0, par), leaf(E0, par)), prob=prob,
                 target=_target(a, c["px"], c["py"], c["pz"], L, rng))
    else:
        s = dict(bf=batch.BatchForward(_batch_mols(c, seed), DEV, want_pps=False, **TIGHT))
    s["case"] = dict(case)
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "grid":
        return D.grid_project(*s["args"], cap=s["cap"], out=s["out"], base=s["base"])
    if k == "scan":
        if c["strokes"]:
            FEs, disps, PPs = D.relax_strokes(s["grid"], s["spec"], s["pts"], c["pz"], [0, 0, -0.1, 0],
                                              s["tip"].stiffness, s["tip"].dpos0, s["tip"].relax, max_iter=100,
                                              f2conv=1e-8, scan_ny=c["py"])
            return {"FEs": FEs, "disps": disps, "PPs": PPs}
        FEs, PPs = D.relax_tilted(s["grid"], s["spec"], s["pts"], c["pz"], s["tip"], max_iter=100, f2conv=1e-8,
                                  scan_ny=c["py"], FEs=s["FEs"], PPs=s["PPs"], df_op=s["op"], df=s["df"])
        return {"FEs": FEs, "PPs": PPs, "df": s["df"]}
    if k == "fdbm":
        st = s["step"]
        Ep = fdbm.pauli_scale_(fdbm.fft_combine(_lib.PPM_FFT_CORRELATE, s["rho"], s["tot"], st, st ** 3), s["A"],
                               s["beta"], 1e-30)
        Ee = fdbm.fft_combine(_lib.PPM_FFT_POISSON_CONVOLVE, s["diff"], fdbm.flip3(s["dlt"]), st,
                              fdbm.POISSON_SCALE * st ** 3)
        Ev = fdbm.dispersion(s["atoms"], s["origin"], st, s["shape"])
        return {"pauli": Ep, "es": Ee, "vdw": Ev, "grid": fdbm.compose_gradient((Ep, Ee, Ev), st)}
    if k == "ewald":
        return s["ew"].tip_grid(s["spec"], *TIPS[c["tip"]], out=s["out"])
    if k in ("fit", "direct"):
        for v in s["leaves"]:
            v.grad = None
        image = (diff.df_image if k == "fit" else diff.direct_df_image)(*s["leaves"], s["prob"])
        loss = 0.5 * ((image - s["target"]) ** 2).sum()
        loss.backward()
        return {"df": image.detach(), "loss": loss.detach(),
                "grads": [v.grad for v in s["leaves"] if v.grad is not None]}
    return s["bf"].forward()


def work(case):
    """Inputs read once, outputs written once; a pair sum counts 20 operations per voxel and site."""
    c, k = case, case["kind"]
    vox = c.get("nx", 0) * c.get("ny", 0) * c.get("nz", 0)
    if k == "grid":
        sites = (c["atoms"] or 16 * c["cells"] ** 2) * (2 * c["npbc"] + 1) ** 2
        return {"bytes": vox * (32.0 if c["base"] else 16.0) + 32.0 * sites, "flops": 20.0 * vox * sites}
    if k == "fdbm":
        return {"bytes": vox * 44.0, "flops": vox * (12.5 * math.log2(vox) + 12.0 * c["atoms"] + 40)}
    if k == "ewald":
        return {"bytes": vox * 16.0, "flops": vox * 64.0}
    if k == "batch":
        st = c["mols"] * c["px"] ** 2 * c["pz"]
        pairs = c["mols"] * 240 ** 2 * 45.0 * 9 * (10 + c["max_atoms"]) / 2
        return {"bytes": st * 20.0 + c["mols"] * 240 ** 2 * 45 * 16.0, "flops": st * 30 * 130.0 + 20 * pairs}
    states = c["px"] * c.get("py", c["px"]) * c["pz"]
    scan = states * 30 * 130.0
    if k == "scan":
        return {"bytes": states * 36.0 + vox * 4.0, "flops": scan}
    if k == "direct":
        return {"bytes": states * 36.0, "flops": states * c["atoms"] * 60.0 * 25}
    win = c["nx"] * c["ny"] * (c["pz"] + 22)
    return {"bytes": win * 48.0 + states * 72.0, "flops": 2 * 20.0 * win * c["atoms"] * 9 + scan}


# ── the same in float64 ───────────────────────────────────────────────────────────────

def _sites(a, npbc, lvA, lvB):
    a = np.asarray(a, np.float64)
    im = [(i, j) for j in range(-npbc, npbc + 1) for i in range(-npbc, npbc + 1)]
    sh = np.array([[i * float(lvA[0]) + j * float(lvB[0]), i * float(lvA[1]) + j * float(lvB[1]), 0] for i, j in im])
    return a[:, None, :3] + sh[None]


def _axes(spec, n=None, k0=0):
    """Voxel coordinates per axis of an axis-aligned spec (planes k0 on for z), float64."""
    nx, ny, nz = spec.n if n is None else n
    f = [float(spec.dA[0]), float(spec.dB[1]), float(spec.dC[2])]
    i = [np.arange(nx), np.arange(ny), k0 + np.arange(nz)]
    return [torch.as_tensor(float(spec.p0[q]) + f[q] * i[q], device=DEV, dtype=torch.float64) for q in range(3)]


def _grid64(axes, a, cp, model, tip, npbc, lvA, lvB, cap, base=None):
    """The force-field grid in float64, (nz,ny,nx,4)."""
    X, Y, Z = axes[0][None, None, :], axes[1][None, :, None], axes[2][:, None, None]
    out = torch.zeros((Z.numel(), Y.numel(), X.numel(), 4), device=DEV, dtype=torch.float64)
    F = [torch.zeros(out.shape[:3], device=DEV, dtype=torch.float64) for _ in range(4)]
    Qs, QZs = TIPS[tip]
    charges = [(float(np.float32(q)) * COULOMB, float(np.float32(z))) for q, z in zip(Qs, QZs) if q]
    cp = np.asarray(cp, np.float64)
    for j, images in enumerate(_sites(a, npbc, lvA, lvB)):
        qa = float(a[j, 3])
        for x, y, z in images:
            dx, dy, dz = X - x, Y - y, Z - z
            dxy2 = dx * dx + dy * dy + R2SAFE
            r2 = dxy2 + dz * dz
            if model == "lj":
                i2 = r2.reciprocal()
                i6 = i2 * i2 * i2
                F[3].add_((cp[j, 1] * i6 - cp[j, 0]).mul_(i6))
                f = (12 * cp[j, 1] * i6 - 6 * cp[j, 0]).mul_(i6).mul_(i2)
            else:
                r = r2.sqrt()
                R0, E0, K = cp[j, :3]
                ex = torch.exp(K * (r - R0))
                F[3].add_(E0 * ex * (ex - 2))
                f = (-2 * K * E0) * ex * (ex - 1) / r
            off = []
            for Q, zo in charges:
                i1 = r2.rsqrt() if zo == 0 else (dxy2 + (dz + zo) ** 2).rsqrt()
                e = (Q * qa) * i1
                F[3].add_(e)
                e = e * i1 * i1
                if zo == 0:
                    f = f + e
                else:
                    off.append((e, zo))
            for e, zo in off:
                F[2].add_(e * (dz + zo))
                F[0].add_(e * dx)
                F[1].add_(e * dy)
            F[0].add_(f * dx)
            F[1].add_(f * dy)
            F[2].add_(f * dz)
    for q in range(4):
        out[..., q] = F[q]
    if base is not None:
        out += base
    if cap:
        out *= (100.0 / out[..., 3:].abs()).clamp(max=1.0)
    return out


class _GridField:
    """Trilinear model of a periodic float64 grid: force, its Jacobian and energy at points (n,3)."""

    def __init__(self, G, spec, k0=0):
        self.G = G.reshape(-1, 4)
        self.n = [int(v) for v in spec.n]
        self.k0, self.nzs = k0, G.shape[0]
        d = [spec.dinvA, spec.dinvB, spec.dinvC]
        self.s = [float(d[q][q]) for q in range(3)]
        self.o = [float(d[q][3]) for q in range(3)]

    def cell(self, p):
        i, w = [], []
        for q in range(3):
            u = p[:, q] * self.s[q] + self.o[q]
            t = (u - u.floor()) * self.n[q] - 0.5
            f = t.floor()
            a = f.long()
            i.append((a % self.n[q], (a + 1) % self.n[q]))
            w.append(t - f)
        k = [(v - self.k0).clamp(0, self.nzs - 1) for v in i[2]]
        idx = [(k[c >> 2] * self.n[1] + i[1][(c >> 1) & 1]) * self.n[0] + i[0][c & 1] for c in range(8)]
        return idx, w

    def __call__(self, p, jac=True):
        idx, (a, b, c) = self.cell(p)
        f = [self.G[i] for i in idx]
        wa, wb, wc = [(1 - a, a)], [(1 - b, b)], [(1 - c, c)]
        A, B, C = wa[0], wb[0], wc[0]
        val = sum((A[m & 1] * B[(m >> 1) & 1] * C[m >> 2])[:, None] * f[m] for m in range(8))
        if not jac:
            return val, None
        sg = (-1.0, 1.0)
        J = torch.stack([
            sum((sg[m & 1] * B[(m >> 1) & 1] * C[m >> 2])[:, None] * f[m] for m in range(8)) * (self.n[0] * self.s[0]),
            sum((A[m & 1] * sg[(m >> 1) & 1] * C[m >> 2])[:, None] * f[m] for m in range(8)) * (self.n[1] * self.s[1]),
            sum((A[m & 1] * B[(m >> 1) & 1] * sg[m >> 2])[:, None] * f[m] for m in range(8)) * (self.n[2] * self.s[2]),
        ], -1)                                              # (n, channel, coordinate)
        return val, J


class _DirectField:
    """The gridless Morse + probe-charge field in float64."""

    def __init__(self, a, R0, E0, K=-1.8):
        t = lambda v: torch.as_tensor(np.asarray(v, np.float64), device=DEV)  # noqa: E731
        self.x, self.q = t(a[:, :3]), t(a[:, 3]) * float(np.float32(W.PROBE_Q)) * COULOMB
        self.R0, self.E0, self.K = t(R0), t(E0), float(np.float32(K))

    def __call__(self, p, jac=True):
        d = p[:, None, :] - self.x[None]
        r = (d.square().sum(-1) + R2SAFE).sqrt()
        ex = torch.exp(self.K * (r - self.R0))
        e1 = 2 * self.K * self.E0 * ex * (ex - 1) - self.q / r ** 2            # dE/dr
        E = (self.E0 * ex * (ex - 2) + self.q / r).sum(1, keepdim=True)
        val = torch.cat([(-(e1 / r)[..., None] * d).sum(1), E], 1)
        if not jac:
            return val, None
        e2 = 2 * self.K ** 2 * self.E0 * ex * (2 * ex - 1) + 2 * self.q / r ** 3
        H = ((e2 - e1 / r) / r ** 2)[..., None, None] * d[..., :, None] * d[..., None, :]
        H = H.sum(1) + (e1 / r).sum(1)[:, None, None] * torch.eye(3, device=DEV, dtype=torch.float64)
        return val, torch.cat([-H, val[:, None, :3]], 1)


def _spring(dp, tip):
    k = [float(v) for v in tip.stiffness]
    d0 = [float(v) for v in tip.dpos0]
    r = dp.norm(dim=1).clamp(min=1e-10)
    eye = torch.eye(3, device=DEV, dtype=torch.float64)
    kv = torch.tensor(k[:3], device=DEV, dtype=torch.float64)
    phi = k[3] * (1 - d0[3] / r)
    g = (dp - torch.tensor(d0[:3], device=DEV, dtype=torch.float64)) * kv + dp * phi[:, None]
    J = eye * kv + phi[:, None, None] * eye + (k[3] * d0[3] / r ** 3)[:, None, None] * dp[:, :, None] * dp[:, None, :]
    return g, J


def _solve3(A, b):
    """Solutions of the 3x3 systems A x = b (n,3,3), (n,3)."""
    c = torch.linalg.cross
    r0, r1, r2 = A[:, :, 0], A[:, :, 1], A[:, :, 2]
    c12, c20, c01 = c(r1, r2), c(r2, r0), c(r0, r1)
    det = (r0 * c12).sum(1)
    return torch.stack([(b * c12).sum(1), (b * c20).sum(1), (b * c01).sum(1)], 1) / det[:, None]


def _eigmin(S):
    """Smallest eigenvalue of symmetric 3x3 matrices (n,3,3), by the trigonometric closed form."""
    q = (S[:, 0, 0] + S[:, 1, 1] + S[:, 2, 2]) / 3
    B = S - q[:, None, None] * torch.eye(3, device=DEV, dtype=torch.float64)
    p = (B.square().sum((1, 2)) / 6).sqrt().clamp(min=1e-300)
    B = B / p[:, None, None]
    det = (B[:, 0] * torch.linalg.cross(B[:, 1], B[:, 2])).sum(1)
    return q + 2 * p * torch.cos(torch.acos((det / 2).clamp(-1, 1)) / 3 + 2 * math.pi / 3)


def _start(pts, tip):
    """Anchors (float32, as they advance), their step and the first probe positions of a descent."""
    anchor = torch.as_tensor(np.asarray(pts, np.float32)[:, :3].copy(), device=DEV)
    step = torch.tensor([0, 0, float(np.float32(tip.tipC[3]))], device=DEV)
    return anchor, step, anchor.double() + torch.as_tensor(np.asarray(tip.dpos0[:3], np.float64), device=DEV)


def _equilibria(field, pts, nz, tip):
    """Probe equilibria of the z descent: (values (n,nz,4), positions (n,nz,3)), by Newton steps on
    the energy (shifted to a positive definite Hessian, at most 0.05 A long)."""
    anchor, step, pos = _start(pts, tip)
    vals, poss = [], []
    for _ in range(nz):
        t = anchor.double()
        for it in range(60):
            v, J = field(pos)
            gs, Js = _spring(pos - t, tip)
            g, H = v[:, :3] + gs, -(J[:, :3] + Js)
            if float(g.abs().max()) < 1e-11:
                break
            lmin = _eigmin(0.5 * (H + H.transpose(1, 2)))
            mu = torch.where(lmin < 1e-3, 0.01 - lmin, torch.zeros_like(lmin))
            d = _solve3(H + mu[:, None, None] * torch.eye(3, device=DEV, dtype=torch.float64), g)
            d *= (0.05 / d.norm(dim=1, keepdim=True).clamp(min=1e-30)).clamp(max=1.0)
            pos = pos + (d if it < 20 else (0.5 if it < 40 else 0.25) * d)
        vals.append(field(pos, jac=False)[0])
        poss.append(pos)
        anchor = anchor + step                                  # the anchors advance in float32
        pos = pos + step.double()
    return torch.stack(vals, 1), torch.stack(poss, 1)


def _fire(field, pts, nz, tip, max_iter, f2conv, strokes):
    """The FIRE descent itself: values (n,nz,4) at the final positions (strokes: before the last
    step) and displacements of the probe from its rest position."""
    anchor, step, pos = _start(pts, tip)
    d0 = torch.as_tensor(np.asarray(tip.dpos0[:3], np.float64), device=DEV)
    n = pos.shape[0]
    dt = torch.full((n,), float(np.float32(tip.relax[0])), device=DEV, dtype=torch.float64)
    damp = torch.full_like(dt, float(np.float32(tip.relax[1])))
    dtmax, damp0 = float(dt[0]), float(damp[0])
    vals, disp = [], []
    for _ in range(nz):
        t = anchor.double()
        v = torch.zeros_like(pos)
        on = torch.ones(n, device=DEV, dtype=torch.bool)
        keep = torch.zeros((n, 4), device=DEV, dtype=torch.float64)
        for it in range(max_iter):
            fe, _ = field(pos, jac=False)
            f = fe[:, :3] + _spring(pos - t, tip)[0]
            ff, vv, vf = f.square().sum(1), v.square().sum(1), (v * f).sum(1)
            keep = torch.where(on[:, None], fe, keep)
            up = vf < 0
            cf = damp * (vv / (ff + 1e-8)).sqrt()
            nv = torch.where(up[:, None], torch.zeros_like(v), v * (1 - damp)[:, None] + f * cf[:, None])
            ndt = torch.where(up, (dt * 0.5).clamp(min=0.1 * dtmax), (dt * 1.1).clamp(max=dtmax))
            nv = nv + f * ndt[:, None]
            damp = torch.where(on, torch.where(up, torch.full_like(damp, damp0), damp * 0.99), damp)
            dt = torch.where(on, ndt, dt)
            v = torch.where(on[:, None], nv, v)
            pos = torch.where(on[:, None], pos + nv * dt[:, None], pos)
            on = on & (ff >= f2conv)
            if it % 8 == 7 and not bool(on.any()):
                break
        vals.append(keep if strokes else field(pos, jac=False)[0])
        disp.append(pos - t - d0)
        anchor = anchor + step
        pos = pos + step.double()
    return torch.stack(vals, 1), torch.stack(disp, 1)


def _giessibl(n, dz, amp=1.0, f0=30000.0, k=1800.0):
    """(n, n) operator: the Giessibl integral of the clamped piecewise-linear Fz column."""
    M = np.zeros((n, n))
    beta = amp / dz
    J1 = lambda u: -math.sqrt(max(0.0, 1 - u * u))  # noqa: E731
    J2 = lambda u: 0.5 * (math.asin(max(-1.0, min(1.0, u))) - u * math.sqrt(max(0.0, 1 - u * u)))  # noqa: E731
    for i in range(n):
        cuts = sorted({-1.0, 1.0, *(u for m in range(-1, n + 1) for u in [(m - i) / beta] if -1 < u < 1)})
        for a, b in zip(cuts[:-1], cuts[1:]):
            cm = i + beta * 0.5 * (a + b)
            d1, d2 = J1(b) - J1(a), J2(b) - J2(a)
            if cm <= 0 or cm >= n - 1:
                M[i, 0 if cm <= 0 else n - 1] += d1
            else:
                j = math.floor(cm)
                M[i, j] += (1 - (i - j)) * d1 - beta * d2
                M[i, j + 1] += (i - j) * d1 + beta * d2
    return torch.as_tensor(-(f0 / (math.pi * k * amp)) * EV_A2_TO_N_M * M, device=DEV)


def _window(spec, zlo, zhi):
    dz, p = float(spec.dC[2]), float(spec.p0[2])
    k0 = max(0, int(math.floor((zlo - p) / dz)) - 1)
    k1 = min(int(spec.n[2]), int(math.ceil((zhi - p) / dz)) + 2)
    return k0, k1 - k0


def _fit_grads(a, cp, R0, E0, G, field, pts, nz, tip, pos, u, spec, k0, npbc, lvA, lvB):
    """Gradients of the loss by the implicit-function theorem: (d xyz, d q, d R0, d E0)."""
    n = pos.shape[0]
    anchors, step, _ = _start(pts, tip)
    gG = torch.zeros_like(G.reshape(-1, 4))
    for iz in range(nz):
        p = pos[:, iz]
        v, J = field(p)
        j = J[:, :3] + _spring(p - anchors.double(), tip)[1]
        ru = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
        ru[:, 2] = u[:, iz]
        lam = _solve3(j.transpose(1, 2), (J[:, :3] * ru[:, :, None]).sum(1))
        idx, w = field.cell(p)
        wt = [(1 - x, x) for x in w]
        for m in range(8):
            gG[:, :3].index_add_(0, idx[m], (wt[0][m & 1] * wt[1][(m >> 1) & 1] * wt[2][m >> 2])[:, None] * (ru - lam))
        anchors = anchors + step
    hit = gG.abs().amax(1).nonzero().ravel()
    g = gG[hit]
    nx, ny = int(spec.n[0]), int(spec.n[1])
    ax = _axes(spec)
    vox = torch.stack([ax[0][hit % nx], ax[1][(hit // nx) % ny], ax[2][k0 + hit // (nx * ny)]], 1)
    Q = float(np.float32(W.PROBE_Q)) * COULOMB
    res = torch.zeros((len(a), 6), dtype=torch.float64)
    for jat, images in enumerate(_sites(a, npbc, lvA, lvB)):
        acc = torch.zeros(6, device=DEV, dtype=torch.float64)
        c6, c12 = float(cp[jat, 0]), float(cp[jat, 1])
        for im in images:
            d = vox - torch.as_tensor(im, device=DEV)
            s = d.square().sum(1) + R2SAFE
            i2 = 1 / s
            i6 = i2 ** 3
            ec = float(a[jat, 3]) * Q * i2.sqrt()
            fr = ((12 * c12 * i6 - 6 * c6) * i6 + ec) * i2
            dfr = ((-84 * c12 * i6 + 24 * c6) * i6 - 1.5 * ec) * i2 * i2
            gd = (g[:, :3] * d).sum(1)
            acc[:3] -= (fr[:, None] * g[:, :3] + (2 * gd * dfr - g[:, 3] * fr)[:, None] * d).sum(0)
            acc[3] += (Q * i2.sqrt() * (gd * i2 + g[:, 3])).sum()
            acc[4] += (-i6 * (6 * gd * i2 + g[:, 3])).sum()
            acc[5] += (i6 * i6 * (12 * gd * i2 + g[:, 3])).sum()
        res[jat] = acc.cpu()
    R, E = (torch.as_tensor(np.asarray(v, np.float64)) for v in (R0, E0))
    dR = res[:, 4] * 12 * E * R ** 5 + res[:, 5] * 12 * E * R ** 11
    dE = res[:, 4] * 2 * R ** 6 + res[:, 5] * R ** 12
    return res[:, :3].to(DEV), res[:, 3].to(DEV), dR.to(DEV), dE.to(DEV)


def _direct_grads(f, a, pts, nz, tip, pos, u):
    """The same for the gridless field."""
    anchors, step, _ = _start(pts, tip)
    th = [f.x.clone(), torch.as_tensor(np.asarray(a[:, 3], np.float64), device=DEV), f.R0.clone(), f.E0.clone()]
    tot = [torch.zeros_like(v) for v in th]
    Q = float(np.float32(W.PROBE_Q)) * COULOMB
    for iz in range(nz):
        p = pos[:, iz]
        _, J = f(p)
        j = J[:, :3] + _spring(p - anchors.double(), tip)[1]
        ru = torch.zeros_like(p)
        ru[:, 2] = u[:, iz]
        w = ru - _solve3(j.transpose(1, 2), (J[:, :3] * ru[:, :, None]).sum(1))
        with torch.enable_grad():
            lv = [v.clone().requires_grad_(True) for v in th]
            h = _DirectField.__new__(_DirectField)
            h.x, h.q, h.R0, h.E0, h.K = lv[0], lv[1] * Q, lv[2], lv[3], f.K
            loss = (h(p, jac=False)[0][:, :3] * w).sum()
            for t, v in zip(tot, torch.autograd.grad(loss, lv)):
                t += v
        anchors = anchors + step
    return tot


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "grid":
        a, cp, lvA, lvB, spec = _grid_inputs(c, seed)
        base = _base_field(c, seed) if c["base"] else None
        return _grid64(_axes(spec), a, cp, c["model"], c["tip"], c["npbc"], lvA, lvB, not c["cells"], base)
    if k == "scan":
        G, spec, L = _scan_grid(c, seed)
        v, d = _fire(_GridField(G.double(), spec), _raster(L, c["px"], c["py"], 12.0), c["pz"], _tip(), 100, 1e-8,
                     c["strokes"])
        if c["strokes"]:
            return {"FEs": v, "disps": torch.cat([d, torch.zeros_like(d[..., :1])], -1), "PPs": None}
        return {"FEs": v, "PPs": None, "df": v[..., 2] @ _giessibl(c["pz"], float(np.float32(-0.1))).T}
    if k == "fdbm":
        s = _fdbm_inputs(c, seed)
        st, n = s["step"], s["shape"]
        fft, ifft = torch.fft.fftn, lambda v: torch.fft.ifftn(v).real  # noqa: E731
        overlap = ifft(fft(s["rho"].double()) * fft(s["tot"].double()).conj()) * st ** 3
        Ep = s["A"] * overlap.clamp(min=1e-30) ** s["beta"]
        kk = [2 * math.pi * torch.fft.fftfreq(m, d=st, device=DEV, dtype=torch.float64) for m in n]
        k2 = kk[0][:, None, None] ** 2 + kk[1][None, :, None] ** 2 + kk[2][None, None, :] ** 2
        k2[0, 0, 0] = math.inf
        es = fft(s["diff"].double()) * fft(s["dlt"].double().flip((0, 1, 2))) / k2
        Ee = ifft(es) * (4 * math.pi * COULOMB * st ** 3)
        ax = [torch.as_tensor(float(np.float32(o)) + float(np.float32(st)) * np.arange(m), device=DEV)
              for o, m in zip(s["origin"], n)]
        Ev = torch.zeros(n, device=DEV, dtype=torch.float64)
        for x, y, z, w in s["atoms"].double().tolist():
            Ev -= w / ((ax[0][:, None, None] - x) ** 2 + (ax[1][None, :, None] - y) ** 2
                       + (ax[2][None, None, :] - z) ** 2 + 2.25) ** 3
        E = Ep + Ee + Ev
        F = [-(E.roll(-1, q) - E.roll(1, q)) / (2 * st) for q in range(3)]
        return {"pauli": Ep, "es": Ee, "vdw": Ev, "grid": torch.stack(F + [E], -1).permute(2, 1, 0, 3).contiguous()}
    if k == "ewald":
        return _ewald64(c, seed)
    if k in ("fit", "direct"):
        a, R0, E0, L, top, rng = _fit_inputs(c, seed)
        pts, tip, nz = _raster(L, c["px"], c["py"], top), _tip(), c["pz"]
        lvA, lvB = np.array([L[0], 0, 0], np.float32), np.array([0, L[1], 0], np.float32)
        target = _target(a, c["px"], c["py"], nz, L, rng).double()
        M = _giessibl(nz, float(np.float32(-0.1)))
        if k == "fit":
            spec, _ = _spec(c, z0=-8.0)
            cp = np.stack([2 * E0.astype(np.float64) * R0.astype(np.float64) ** 6,
                           E0.astype(np.float64) * R0.astype(np.float64) ** 12], 1)
            k0, kn = _window(spec, top - 4.0 - 0.1 * (nz - 1) - 1.0, top - 4.0 + 1.0)
            G = _grid64(_axes(spec, (spec.n[0], spec.n[1], kn), k0), a, cp, "lj", "point", 1, lvA, lvB, True)
            field = _GridField(G, spec, k0)
        else:
            field = _DirectField(a, R0, E0)
        v, pos = _equilibria(field, pts, nz, tip)
        img = v[..., 2] @ M.T
        r = img - target.reshape(img.shape)
        u = r @ M
        if k == "fit":
            gr = _fit_grads(a, cp, R0, E0, G, field, pts, nz, tip, pos, u, spec, k0, 1, lvA, lvB)
            gr = list(gr if c["params"] else gr[:2])
        else:
            gr = _direct_grads(field, a, pts, nz, tip, pos, u)
        return {"df": img.reshape(c["px"], c["py"], nz), "loss": 0.5 * (r * r).sum(), "grads": gr}
    out = []
    for w in _batch_mols(c, seed):
        spec = D.axis_aligned_spec(w.p0, w.L, w.n)
        zt = float(w.scan_p0[2])
        k0, kn = _window(spec, zt - 4.0 - 0.1 * (w.nz - 1) - 0.4, zt - 4.0 + 0.6)
        G = _grid64(_axes(spec, (spec.n[0], spec.n[1], kn), k0), w.atoms, w.cLJ, "lj", "point", 1, w.lvA, w.lvB, True)
        v, _ = _equilibria(_GridField(G, spec, k0), D.scan_points(w.scan_p0, w.scan_da, w.scan_db, *w.nxy), w.nz,
                           _tip())
        out.append(v[..., 2] @ _giessibl(w.nz, float(np.float32(-0.1))).T)
    return torch.cat(out)


def _ewald64(c, seed):
    """Probe field of the slab from the reciprocal series over every G up to n_harm."""
    ions, Lxy, spec = _ewald_inputs(c, seed)
    ax = _axes(spec)
    t = lambda v: torch.as_tensor(np.asarray(v, np.float64), device=DEV)  # noqa: E731
    x, y, z, q = (t(ions[:, i]) for i in range(4))
    n = c["n_harm"]
    h, kk = torch.meshgrid(torch.arange(-n, n + 1, device=DEV), torch.arange(-n, n + 1, device=DEV), indexing="ij")
    h, kk = h.ravel().double(), kk.ravel().double()
    keep = (h > 0) | ((h == 0) & (kk > 0))                 # each entry stands for the pair +-G
    b = 2 * math.pi / Lxy
    gx, gy = h[keep] * b, kk[keep] * b
    gn = torch.hypot(gx, gy)
    zl = torch.unique(z)
    S = torch.stack([(q[z == v] * torch.exp(-1j * (gx[:, None] * x[z == v] + gy[:, None] * y[z == v]))).sum(1)
                     for v in zl])
    S = S * (4 * math.pi / (Lxy * Lxy * gn))
    big = S.abs().amax(0)
    sel = big > 1e-9 * big.max()
    gx, gy, gn, S = gx[sel], gy[sel], gn[sel], S[:, sel]
    out = torch.zeros((c["nz"], c["ny"], c["nx"], 4), device=DEV, dtype=torch.float64)
    ql = torch.stack([q[z == v].sum() for v in zl])
    Qs, QZs = TIPS[c["tip"]]
    T = torch.zeros((c["nz"], gx.numel()), device=DEV, dtype=torch.complex128)
    dT = torch.zeros_like(T)
    t0 = torch.zeros((c["nz"], 2), device=DEV, dtype=torch.float64)
    for Q, zo in zip(Qs, QZs):
        if not Q:
            continue
        Q = float(np.float32(Q)) * COULOMB
        d = ax[2][:, None] + float(np.float32(zo)) - zl[None]
        for l in range(len(zl)):
            e = Q * torch.exp(-gn[None] * d[:, l:l + 1].abs())
            T += e * S[l]
            dT += -torch.sign(d[:, l:l + 1]) * gn[None] * e * S[l]
        t0[:, 0] -= Q * 2 * math.pi / (Lxy * Lxy) * (ql * d.abs()).sum(1)
        t0[:, 1] -= Q * 2 * math.pi / (Lxy * Lxy) * (ql * torch.sign(d)).sum(1)
    ey = torch.exp(1j * gy[:, None] * ax[1][None])
    ex = torch.exp(1j * gx[:, None] * ax[0][None])
    for iz in range(c["nz"]):
        P = [((v[iz][:, None] * ey).T @ ex) for v in (T, T * (1j * gx), T * (1j * gy), dT)]
        out[iz, ..., 3] = P[0].real + t0[iz, 0]
        out[iz, ..., 0], out[iz, ..., 1] = -P[1].real, -P[2].real
        out[iz, ..., 2] = -P[3].real - t0[iz, 1]
    return out
