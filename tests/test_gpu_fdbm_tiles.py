"""The force grid's tiles and the dispersion's voxels per thread at their edges.

compose_gradient: the sums, differences and quotients of each voxel are single FP32 operations in a fixed order, so
NumPy's float32 gives the same bits.  Dispersion: 1e-5 relative per voxel against FP64, the bar of
test_gpu_fdbm.py, over both numbers of voxels per thread; and denominators at both ends of the short reciprocal's
range (an atom on a voxel with RA = 0, a position whose square overflows), where the quotient is IEEE's.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from spammm_amd import device as D      # noqa: E402
from spammm_amd import fdbm             # noqa: E402


@pytest.mark.parametrize("nf", [1, 2, 3])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 2), (16, 3, 16), (17, 2, 15), (15, 9, 17), (33, 5, 40), (3, 8, 64)])
def test_compose_gradient_bits(shape, nf):
    rng = np.random.default_rng(2)
    f = [rng.normal(size=shape).astype(np.float32) for _ in range(nf)]
    step = 0.13
    dev = D.require_gpu()
    g = fdbm.compose_gradient(tuple(torch.as_tensor(v, device=dev) for v in f), step).cpu().numpy()
    E = np.zeros(shape, np.float32)
    for v in f:
        E = E + v
    h2 = np.float32(2.0) * np.float32(step)
    want = np.stack([-(np.roll(E, -1, a) - np.roll(E, 1, a)) / h2 for a in range(3)] + [E], -1)
    np.testing.assert_array_equal(g.reshape(shape[::-1] + (4,)), want.transpose(2, 1, 0, 3))


@pytest.mark.parametrize("shape", [(1, 3, 5), (30, 31, 33), (83, 80, 80), (81, 79, 85)])     # from 524,288 voxels: 4 a thread
def test_dispersion_voxels_per_thread(shape):
    rng = np.random.default_rng(4)
    step, RA, org = 0.15, 1.5, np.array([-1.0, 0.5, 2.0])
    at = np.concatenate([rng.uniform(0, 9, (300, 3)), rng.uniform(5, 40, (300, 1))], 1).astype(np.float32)
    dev = D.require_gpu()
    got = fdbm.dispersion(torch.as_tensor(at, device=dev), org, step, shape, RA).cpu().numpy().astype(np.float64)
    pick = rng.integers(0, np.prod(shape), 2000)
    pick[:2] = 0, np.prod(shape) - 1
    idx = np.stack(np.unravel_index(pick, shape), 1)
    p = org + np.float64(np.float32(step)) * idx
    d2 = ((p[:, None] - at[None, :, :3].astype(np.float64)) ** 2).sum(-1)
    want = -(at[:, 3].astype(np.float64) / (d2 + RA * RA) ** 3).sum(1)
    rel = np.abs(got.reshape(-1)[pick] / want - 1).max()
    print(f"[dispersion] {shape}: max rel err {rel:.2e}")
    assert rel <= 1e-5
    base = torch.randn(shape, device=dev)
    acc = fdbm.dispersion(torch.as_tensor(at, device=dev), org, step, shape, RA, out=base.clone(), accumulate=True)
    assert torch.equal(acc, base + torch.as_tensor(got.astype(np.float32), device=dev).reshape(shape))


@pytest.mark.parametrize("shape", [(5, 4, 6), (83, 80, 80)])
def test_dispersion_denominators_out_of_the_short_range(shape):
    at = np.array([[0.5, 0.25, 0.75, 3.0], [1e25, 0, 0, 7.0], [0.1, 0.1, -2.0, 1.0]], np.float32)
    dev = D.require_gpu()
    got = fdbm.dispersion(torch.as_tensor(at, device=dev), (0., 0., 0.), 0.25, shape, 0.0).cpu().numpy()
    assert got[2, 1, 3] == -np.inf
    got[2, 1, 3] = 0
    assert np.isfinite(got).all()
    p = np.array([1.0, 0.75, 1.0])
    want = -sum(float(a[3]) / ((p - a[:3].astype(np.float64)) ** 2).sum() ** 3 for a in at[[0, 2]])
    assert abs(got[4, 3, 4] / want - 1) <= 1e-5
