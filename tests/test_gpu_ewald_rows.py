"""The slab's probe grid by rows along the lattice vector a: tiles of 32 voxels and 8 rows, pieces of the sum over
k, h left out below the rounding, against the FP64 oracle, and against the form for any grid direction, which takes
the same voxels when the grid's first axis is turned to y.

Tolerance 2e-5 of the largest magnitude, that of the FP32 tables in test_gpu_ewald.py.
"""
import numpy as np
import pytest

from oracle import ewald_ref as E
from tests.test_gpu_ewald import _close, _skew_slab

pytestmark = pytest.mark.gpu


def _grid(ew, n, p0, dA, dB, dz, Qs, QZs, **kw):
    from spammm_amd import device as D
    v = [np.asarray(d, np.float32) for d in (dA, dB, (0, 0, dz))]
    L = np.array([d * m for d, m in zip(v, n)], np.float64)
    spec = D.GridSpec(n, np.asarray(p0, np.float32), *v, *D.dinv_lvec(np.linalg.inv(L).T, n))
    return spec, ew.tip_grid(spec, Qs, QZs, **kw)


@pytest.mark.parametrize("n,n_harm,step", [
    ((1, 1, 1), 1, 0.3),            # one voxel, one h
    ((31, 7, 3), 1, 0.2),           # below a tile and a group of rows
    ((33, 9, 2), 5, 0.17),          # one past them
    ((64, 8, 5), 8, 0.1),           # exactly full
    ((257, 17, 2), 12, 0.05),       # one pair of tiles for each wave and one voxel more
    ((70, 10, 3), 31, 0.07),        # 32 h: every lane of a row
    ((40, 9, 2), 40, 0.11),         # more pieces than lanes
    ((34, 9, 2), 63, 0.13),         # the most h
    ((34, 9, 2), 64, 0.13),         # one more: the form for any direction
])
def test_rows_against_the_oracle_and_the_general_form(n, n_harm, step):
    import torch
    from spammm_amd.ewald import SurfaceEwald
    ions, a, b = _skew_slab(5)
    Qs, QZs = np.array([-0.1, 0.05, 0.0, 0.0]), np.array([0.0, 0.3, 0.0, 0.0])
    ew = SurfaceEwald().prepare_system(ions, a, b, n_harm=n_harm)
    p0, dz = (0.4, -0.7, 0.9), 0.8
    spec, g = _grid(ew, n, p0, (step, 0, 0), (0, 0.9 * step, 0), dz, Qs, QZs)
    o = E.Slab(ions.astype(np.float64), a, b, n_harm)
    ref = E.tip_grid(o, spec.p0.astype(np.float64), np.array([spec.dA[0], spec.dB[1], spec.dC[2]], np.float64), n, Qs,
                     QZs)
    G = g.cpu().numpy().astype(np.float64)
    _, t = _grid(ew, (n[1], n[0], n[2]), p0, (0, 0.9 * step, 0), (step, 0, 0), dz, Qs, QZs)
    T = t.cpu().numpy().astype(np.float64).transpose(0, 2, 1, 3)
    scale = np.abs(ref[..., :3]).max()
    for c, name in enumerate(("Fx", "Fy", "Fz", "E")):
        _close(G[..., c], ref[..., c], 2e-5 * max(1.0, scale / np.abs(ref[..., c]).max()), f"rows {name}")
        _close(T[..., c], ref[..., c], 2e-5 * max(1.0, scale / np.abs(ref[..., c]).max()), f"any direction {name}")
    base = torch.randn(g.shape, dtype=torch.float32, device="cuda")
    _, acc = _grid(ew, n, p0, (step, 0, 0), (0, 0.9 * step, 0), dz, Qs, QZs, out=base.clone(), accumulate=True)
    assert torch.equal(acc, base + g)
