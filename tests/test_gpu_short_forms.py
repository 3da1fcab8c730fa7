"""The short correctly rounded FP32 forms against IEEE's over the mantissas, through the entry points that use them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import oracle as O              # noqa: E402
from spammm_amd import device as D, fdbm    # noqa: E402


def test_reciprocal_over_16_million_operands():
    """One atom, RA = 0, 4096 x 4096 voxels in its xy plane, 2^-6 apart and at whole multiples of 2^-14 from it: the operand
    is RN(x^2 + RN(y^2)), whose sum FP64 holds exactly, and the result -(1/r^2)^3 in three roundings, so NumPy's float32
    gives the same bits if the reciprocal is correctly rounded."""
    n = 4096
    dev = D.require_gpu()
    step, ax, ay = 2.0 ** -6, -85 * 2.0 ** -14, -37 * 2.0 ** -14
    at = torch.tensor([[ax, ay, 0., 1.]], device=dev)
    got = fdbm.dispersion(at, (0., 0., 0.), step, (n, n, 1), 0.0).cpu().numpy().reshape(n, n)
    k = step * np.arange(n)
    y2 = ((k - ay) ** 2).astype(np.float32).astype(np.float64)
    r2 = ((k - ax)[:, None] ** 2 + y2[None]).astype(np.float32)
    i = np.float32(1) / r2
    assert len(np.unique(r2.view(np.uint32) & 0x7fffff)) > 4_000_000          # of 2^23 mantissas
    np.testing.assert_array_equal(got, -(i * i * i))


@pytest.mark.parametrize("lanes", [1, 4])
def test_roots_and_quotients_of_millions_of_steps(lanes):
    """12 FIRE steps of 3 heights over 256 x 256 points on a rough grid: 7 million roots, quotients and ratios with as many
    different operands, and a wrong last bit of one stays in its point's result: bit for bit against the FP32 oracle."""
    n = (48, 48, 48)
    rng = np.random.default_rng(5)
    g = rng.normal(0, 0.3, n + (4,)).astype(np.float32)
    sp = D.axis_aligned_spec([-4, -4, -4], [8, 8, 8], n)
    tip = D.Tip(stiffness=np.array([-0.03, -0.04, -0.03, -1.2], np.float32),
                dpos0=np.array([0.2, -0.1, -1.7, 1.7], np.float32), tipC=np.array([0, 0, 1, -0.13], np.float32))
    pts = D.scan_points([-4, -4, 2.0], [8 / 256, 0, 0], [0, 8 / 256, 0], 256, 256)
    FEs, PPs = D.relax_tilted(torch.as_tensor(g, device=D.require_gpu()), sp, torch.as_tensor(pts, device=D.require_gpu()), 3,
                              tip, 12, 1e-30, lanes=lanes)
    FEo, PPo = O.relax_tilted(g, sp.n, sp.dinvA, sp.dinvB, sp.dinvC, pts, 3, tip.tipA, tip.tipB, tip.tipC, tip.stiffness,
                              tip.dpos0, tip.relax, tip.surfFF, 12, 1e-30, False, "f32")
    np.testing.assert_array_equal(PPs.cpu().numpy(), PPo)
    np.testing.assert_array_equal(FEs.cpu().numpy(), FEo)
