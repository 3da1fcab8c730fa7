"""The interpolated grid adjoint: blocks' cotangents gathered at Chebyshev nodes for the far sites, against the pair
laws' adjoint in FP64 at the voxels' FP32 positions.

Tolerance per atom and column: 5e-6 of the sum of the absolute contributions.  FP32 differences of positions carry
1e-7 of a distance and enter the steepest term (r^-14) 14-fold; the terms' own roundings and the interpolation
(below 1e-6 of a term at 12.5 half-widths) come on top.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from spammm_amd import _lib             # noqa: E402
from spammm_amd import device as D      # noqa: E402

COULOMB = 14.3996448915
R2SAFE = 1e-4


def reference(at, cp, spec, Qs, QZs, cot, npbc, lvA, lvB, model):
    """(gradient, sum of absolute contributions), each (na, 6)."""
    dev = cot.device
    idx = (cot != 0).any(-1).nonzero()
    f = lambda v: torch.as_tensor(np.asarray(v, np.float32), device=dev)     # noqa: E731
    i = idx.flip(1).float()
    P = (f(spec.p0)[None] + i[:, :1] * f(spec.dA) + i[:, 1:2] * f(spec.dB) + i[:, 2:] * f(spec.dC)).double()
    G = cot[idx[:, 0], idx[:, 1], idx[:, 2]].double()
    at, cp = at.double(), cp.double()
    g, s = (torch.zeros((len(at), 6), dtype=torch.float64, device=dev) for _ in range(2))

    def put(j, c, v):
        g[j, c] += v.sum(0)
        s[j, c] += v.abs().sum(0)

    def xyz(j, d, fr, dfr):
        put(j, slice(0, 3), -(fr[:, None] * G[:, :3] + (2 * (G[:, :3] * d).sum(1) * dfr - G[:, 3] * fr)[:, None] * d))

    for j in range(len(at)):
        for iy in range(-npbc, npbc + 1):
            for ix in range(-npbc, npbc + 1):
                d = P - (at[j, :3] + ix * f(lvA).double() + iy * f(lvB).double())
                r2 = (d * d).sum(1) + R2SAFE
                gF = (G[:, :3] * d).sum(1)
                if model == _lib.PPM_MODEL_LJ:
                    c6, c12 = cp[j, 0], cp[j, 1]
                    i6 = r2 ** -3
                    xyz(j, d, (12 * c12 * i6 - 6 * c6) * i6 / r2, (-84 * c12 * i6 + 24 * c6) * i6 / r2 ** 2)
                    put(j, 4, -i6 * (6 * gF / r2 + G[:, 3]))
                    put(j, 5, i6 * i6 * (12 * gF / r2 + G[:, 3]))
                else:
                    R0, E0, K = cp[j, 0], cp[j, 1], cp[j, 2]
                    r = r2.sqrt()
                    ex = torch.exp(K * (r - R0))
                    xyz(j, d, -2 * K * E0 * ex * (ex - 1) / r, -K * E0 * ex * (K * (2 * ex - 1) / r - (ex - 1) / r2) / r)
                    put(j, 4, gF * 2 * K * K * E0 * ex * (2 * ex - 1) / r - G[:, 3] * 2 * K * E0 * ex * (ex - 1))
                    put(j, 5, -gF * 2 * K * ex * (ex - 1) / r + G[:, 3] * ex * (ex - 2))
                for Q, zo in zip(Qs, QZs):
                    if Q:
                        do = d + torch.tensor([0., 0., np.float32(zo)], dtype=torch.float64, device=dev)
                        ro = (do * do).sum(1) + R2SAFE
                        e = float(np.float32(Q)) * COULOMB * ro ** -.5
                        xyz(j, do, at[j, 3] * e / ro, -1.5 * at[j, 3] * e / ro ** 2)
                        put(j, 3, G[:, 3] * e + (G[:, :3] * do).sum(1) * e / ro)
    return g, s


CASES = {
    # n, atoms, npbc, lattice edge (0: the grid's), model, Qs, QZs, capped voxels, atoms within
    "ragged_blocks": ((171, 163, 149), 80, 1, 0, "lj", [-.1, 0, 0, 0], [0, 0, 0, 0], 0, 0),
    "capped_blocks": ((176, 160, 160), 80, 1, 0, "lj", [-.1, 0, 0, 0], [0, 0, 0, 0], 6, 0),
    "offset_charges": ((171, 163, 149), 80, 1, 0, "lj", [.05, -.1, .05, 0], [.3, 0, -.3, 0], 0, 0),
    "morse": ((171, 163, 149), 80, 1, 0, "morse", [-.1, 0, 0, 0], [0, 0, 0, 0], 0, 0),
    "near_list_in_parts": ((100, 90, 70), 700, 1, 60, "lj", [0, 0, 0, 0], [0, 0, 0, 0], 0, 5),
}


@pytest.mark.parametrize("name", CASES)
def test_interpolated_adjoint_against_fp64(name):
    n, na, npbc, cell, law, Qs, QZs, ncap, within = CASES[name]
    rng = np.random.default_rng(8)
    dev = D.require_gpu()
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v, np.float32), device=dev)      # noqa: E731
    L = np.array(n) * 0.1
    a = np.zeros((na, 4))
    a[:, :2] = rng.uniform(0, 1, (na, 2)) * (within or L[:2])
    a[:, 2] = rng.uniform(-.5, 0, na) - (4 if within else 0)
    a[:, 3] = rng.uniform(-.3, .3, na)
    model = _lib.PPM_MODEL_LJ if law == "lj" else _lib.PPM_MODEL_MORSE
    cp = (np.stack([rng.uniform(10, 40, na), rng.uniform(1e4, 4e4, na)], 1) if law == "lj" else
          np.stack([rng.uniform(3, 4, na), rng.uniform(.002, .01, na), np.full(na, -1.8), np.zeros(na)], 1))
    spec = D.axis_aligned_spec([0, 0, -2.], L, n)
    lvA, lvB = [cell or L[0], 0, 0], [0, cell or L[1], 0]
    cot = torch.zeros((n[2], n[1], n[0], 4), device=dev)
    k0 = 22 if within else 52
    cot[k0:k0 + 43] = t(rng.normal(size=(43, n[1], n[0], 4)))
    cot[:, 40:44, 30:50] = 0                                   # columns left out inside a block
    grid = torch.zeros_like(cot)
    for _ in range(ncap):                                      # their raw sums are small: differentiated as they are
        grid[k0 + rng.integers(0, 43), rng.integers(0, 40), rng.integers(0, n[0]), 3] = 100.0
    A, C = t(a), t(cp)
    args = (A, C, model, spec, Qs, QZs, grid, cot, (npbc, npbc), lvA, lvB)
    got = D.grid_adjoint(*args, cap=True, params=True)
    part = D.grid_adjoint(*args, cap=True, params=False)
    want, total = reference(A, C, spec, Qs, QZs, cot, npbc, lvA, lvB, model)
    ratio = ((got.to(dev) - want).abs() / total.clamp_min(1e-300)).amax(0)
    print(f"[{name}] error / sum of |contributions| by column:", " ".join(f"{v:.1e}" for v in ratio.tolist()))
    assert (ratio <= 5e-6).all()
    first = ((part.to(dev) - want).abs() / total.clamp_min(1e-300)).amax(0)[:4]      # params = 0: the same bound
    assert (first <= 5e-6).all() and not part[:, 4:].any()
