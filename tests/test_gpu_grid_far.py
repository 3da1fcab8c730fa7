"""GPU: the interpolated grid projection (near sites at the voxels, the others at block nodes) at the
edges of its blocks, levels and lists, against the FP64 oracle; windows and voxel counts per thread."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import oracle as O                                     # noqa: E402
from spammm_amd import device as D, workloads as W                # noqa: E402
from spammm_amd.params import ELEMENTS_BENCH, mix_R0E0, mix_lj    # noqa: E402

TIPS = {"q0": ([W.PROBE_Q, 0, 0, 0], [0, 0, 0, 0]), "offsets": ([0, -0.1, 0.1, 0], [0, 1.8, 3.6, 0]),
        "none": ([0, 0, 0, 0], [0, 0, 0, 0])}

# (name, model, atoms, npbc, voxels, step, tip, skew): one level (few sites or a Morse law) and two
# levels (many sites, >= 150 blocks of 32^3), whole blocks and remainders of 1 and 15 voxels, more sites
# near a workgroup than its list of 512 holds, a sheared x,y cell
CASES = [
    ("one_level", 0, 18, 1, (130, 97, 95), 0.1, "q0", 0.0),
    ("one_level_lj_only", 0, 30, 1, (97, 161, 64), 0.1, "none", 0.0),
    ("one_level_offsets", 0, 60, 0, (176, 161, 145), 0.1, "offsets", 0.0),
    ("one_level_morse", 1, 40, 1, (113, 112, 81), 0.12, "q0", 0.0),
    ("one_level_lists", 0, 100, 1, (100, 90, 70), 0.1, "q0", 0.0),
    ("two_levels", 0, 120, 1, (193, 207, 161), 0.1, "q0", 0.0),
    ("two_levels_lists", 0, 200, 1, (161, 165, 170), 0.1, "q0", 0.0),
    ("two_levels_lj_only_skew", 0, 120, 1, (224, 193, 129), 0.09, "none", 0.3),
    ("two_levels_fine_offsets", 0, 90, 1, (257, 260, 90), 0.05, "offsets", 0.0),
]


def setup(model, na, npbc, n, step, tip, skew, seed=5):
    rng = np.random.default_rng(seed)
    en, pos = W.flake_geometry(na, rng)
    atoms = np.zeros((na, 4), np.float32)
    atoms[:, :3] = pos
    q = rng.uniform(-0.3, 0.3, na)
    atoms[:, 3] = q - q.mean()
    if model == 0:
        cp = mix_lj(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
    else:
        R0, E0 = mix_R0E0(en, ELEMENTS_BENCH, W.PROBE_R0, W.PROBE_E0)
        cp = np.stack([R0, E0, np.full(na, -1.8), np.zeros(na)], 1).astype(np.float32)
    dA, dB, dC = (np.array(v, np.float32) for v in ((step, 0, 0), (skew * step, step, 0), (0, 0, step)))
    L = np.array([dA * n[0], dB * n[1], dC * n[2]], np.float64)
    p0 = np.array([-L[0, 0] / 2 - L[1, 0] / 2, -L[1, 1] / 2, -2.0], np.float32)
    sp = D.GridSpec(n, p0, dA, dB, dC, *D.dinv_lvec(np.linalg.inv(L).T, n))
    lv = [np.asarray(v, np.float32) for v in (L[0], L[1])]
    return atoms, np.ascontiguousarray(cp, np.float32), sp, *TIPS[tip], (npbc, npbc), *lv


def project(s, **kw):
    atoms, cp, sp, Qs, QZs, npbc, lvA, lvB = s
    d = D.require_gpu()
    return D.grid_project(torch.as_tensor(atoms, device=d), torch.as_tensor(cp, device=d),
                          0 if cp.shape[1] == 2 else 1, sp, Qs, QZs, npbc, lvA, lvB, **kw)


def edge_voxels(n, rng, k=1500):
    """Flat indices, half of them on the first or last voxel of a block of 16 along some axis."""
    i = np.stack([rng.integers(0, m, k) for m in n], 1)
    ax = rng.integers(0, 3, k // 2)
    lim = np.asarray(n)[ax]
    i[np.arange(k // 2), ax] = np.minimum(16 * rng.integers(0, lim // 16 + 1) + rng.choice([0, 15], k // 2), lim - 1)
    return (i[:, 2] * n[1] + i[:, 1]) * n[0] + i[:, 0], i


def oracle_at(model, atoms, cp, P, Qs, QZs, npbc, lvA, lvB):
    """FP64 values (k,4) of the pair laws at points P (k,3) float32, from atom images at FP32 positions:
    a one-voxel grid at each point."""
    z = np.zeros(3)
    one = np.zeros(1, np.int64)
    f = np.float32
    im = [(f(i), f(j)) for j in range(-npbc[1], npbc[1] + 1) for i in range(-npbc[0], npbc[0] + 1)]
    sites = np.concatenate([np.c_[(atoms[:, :3] + i * lvA) + j * lvB, atoms[:, 3:]] for i, j in im]).astype(f)
    cps = np.tile(cp, (len(im), 1))
    return np.concatenate([O.grid_voxels(model, sites, cps, (1, 1, 1), p, z, z, z, Qs, QZs, one) for p in P])


def voxel_points(sp, i):
    """Voxel positions (k,3) float32 in the kernels' order of operations."""
    f = np.asarray(i, np.float32)
    p0, dA, dB, dC = (np.asarray(v, np.float32)[:3] for v in (sp.p0, sp.dA, sp.dB, sp.dC))
    return ((p0 + dA * f[:, :1]) + dB * f[:, 1:2]) + dC * f[:, 2:]


@pytest.mark.parametrize("acc64", [False, True])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_interpolated_grid_vs_oracle(case, acc64):
    """Against the FP64 pair laws at the FP32 positions of voxels and images, within the bar of the direct sum: 1e-5 |(F,E)|
    + 4e-6 sum|charge terms| + 1e-6, and without charges 4e-5 |(F,E)| + 1e-9 (a position off by 1e-6 A
    changes a near pair's force by 14/r of itself per A, r >= 0.5 A outside the rescaled voxels)."""
    name, model, na, npbc, n, step, tip, skew = case
    s = setup(model, na, npbc, n, step, tip, skew)
    atoms, cp, sp, Qs, QZs, npb, lvA, lvB = s
    idx, i = edge_voxels(n, np.random.default_rng(1))
    G = project(s, acc64=acc64).cpu().numpy().reshape(-1, 4)
    assert np.isfinite(G).all()
    Go = oracle_at(model, atoms, cp, voxel_points(sp, i), Qs, QZs, npb, lvA, lvB)
    mag = np.linalg.norm(Go, axis=1)
    err = np.abs(G[idx].astype(np.float64) - Go).max(1)
    if tip == "none":
        bound = 4e-5 * mag + 1e-9
    else:
        P = np.asarray(sp.p0, np.float64) + i @ np.array([sp.dA, sp.dB, sp.dC], np.float64)
        S = sum(O.abs_term_sums(atoms, np.zeros((na, 2)), q, npb, lvA, lvB, P + [0, 0, z]) for q, z in zip(Qs, QZs) if q)
        bound = 1e-5 * mag + 4e-6 * S * np.minimum(1.0, 100.0 / np.maximum(np.abs(Go[:, 3]), 1e-300)) + 1e-6
    print(f"[far] {name} acc64={acc64}: worst |d|/bound {(err / bound).max():.3e}", flush=True)
    assert (err <= bound).all()


@pytest.mark.parametrize("name", ["one_level_morse", "two_levels", "two_levels_lists"])
def test_windows_and_base_of_interpolated_grids(name):
    """Any planes of a window carry the whole grid's bits (blocks are aligned to plane 0, whatever a
    launch stores), and a base grid adds to the raw sum before the rescale."""
    s = setup(*next(c for c in CASES if c[0] == name)[1:])
    n = s[2].n
    whole = project(s)
    for klo, nzw in ((0, 1), (15, 2), (16, 16), (31, 33), (5, n[2] - 5), (n[2] - 1, 1)):
        assert torch.equal(project(s, window=(klo, nzw)), whole[klo:klo + nzw]), (klo, nzw)
    raw = project(s, cap=False)
    base = torch.linspace(-0.2, 0.3, raw.numel(), device=raw.device).reshape(raw.shape)
    want = raw + base
    want = want * (100.0 / want[..., 3:].abs()).clamp(max=1.0)
    got = project(s, base=base)
    assert ((got - want).abs() <= 2e-6 * want.abs().amax(-1, keepdim=True)).all()


def test_one_voxel_per_thread_of_small_direct_launches():
    """A directly summed grid (few sites): windows of few workgroups take one voxel per thread and have
    the bits of the whole grid's 8."""
    s = setup(0, 20, 0, (200, 200, 60), 0.1, "q0", 0.0)
    whole = project(s)
    for klo, nzw in ((0, 1), (3, 9), (20, 40)):
        assert torch.equal(project(s, window=(klo, nzw)), whole[klo:klo + nzw]), (klo, nzw)
