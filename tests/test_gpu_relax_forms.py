"""The short FP32 roots and quotients of the relaxation at the ends of their ranges, and the splits of the
direct pair sum.

The relaxation takes the IEEE forms where an operand leaves the middle of the exponent range, on the host's
word (a spring whose rest position is the anchor) or for the columns that meet one: both against the FP32
oracle, bit for bit.  The direct sum's bits depend on its G running sums and not on the lanes that hold
them: a launch with two sums in a lane against a smaller one of the same G with one, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import oracle as O          # noqa: E402
from spammm_amd import device as D      # noqa: E402
from spammm_amd import workloads as W   # noqa: E402
from tests.test_gpu_parity import dev, grid_gpu, tip_of   # noqa: E402

# name: scale of the force grid (left half, right half in x), spring at rest on the anchor, spring off
FORMS = {
    "ordinary": (1.0, 1.0, False, False),
    "rest_at_anchor": (1.0, 1.0, True, False),
    "no_field": (0.0, 0.0, False, False),
    "tiny_forces_free_tip": (1e-18, 1e-18, False, True),
    "huge_forces": (1e12, 1e12, False, False),
    "tiny_and_ordinary_columns": (1e-18, 1.0, False, True),
    "huge_and_ordinary_columns": (1e12, 1.0, False, False),
}


@pytest.mark.parametrize("lanes", [1, 2, 4])
@pytest.mark.parametrize("form", FORMS)
def test_relaxation_bits_at_the_ends_of_the_ranges(form, lanes):
    left, right, anchor, free = FORMS[form]
    w = W.small()
    G, sp = grid_gpu(w)
    G = G.clone()
    half = G.shape[2] // 2
    G[:, :, :half] *= left
    G[:, :, half:] *= right
    g = G.cpu().numpy()
    tip = tip_of(w)
    if anchor:
        tip.dpos0 = np.zeros(4, np.float32)
    if free:
        tip.stiffness = np.zeros(4, np.float32)
    pts = D.scan_points(w.scan_p0, w.scan_da, w.scan_db, *w.nxy)
    P = torch.as_tensor(pts, device=dev())
    for cb in (True, False):
        FEs, PPs = D.relax_tilted(G, sp, P, w.nz, tip, 12, 1e-30, check_before=cb, lanes=lanes)
        FEo, PPo = O.relax_tilted(g, sp.n, sp.dinvA, sp.dinvB, sp.dinvC, pts, w.nz, tip.tipA, tip.tipB, tip.tipC,
                                  tip.stiffness, tip.dpos0, tip.relax, tip.surfFF, 12, 1e-30, cb, "f32")
        np.testing.assert_array_equal(PPs.cpu().numpy(), PPo)
        np.testing.assert_array_equal(FEs.cpu().numpy(), FEo)
    dTip = np.array([0., 0., -0.1, 0.], np.float32)
    FEs, disps, PPs = D.relax_strokes(G, sp, P, w.nz, dTip, tip.stiffness, tip.dpos0, tip.relax, 12, 1e-30)
    FEo, dio, PPo = O.relax_strokes(g, sp.n, sp.dinvA, sp.dinvB, sp.dinvC, pts, w.nz, dTip, tip.stiffness, tip.dpos0,
                                    tip.relax, 12, 1e-30, "f32")
    np.testing.assert_array_equal(PPs.cpu().numpy(), PPo)
    np.testing.assert_array_equal(FEs.cpu().numpy(), FEo)
    np.testing.assert_array_equal(disps.cpu().numpy(), dio)


@pytest.mark.parametrize("na", [128, 100, 65, 33])
@pytest.mark.parametrize("n_many,n_few", [(64, 50), (85, 70)])     # G = 64 and 32 (33 atoms: 32), two sums | one
def test_direct_sum_bits_do_not_depend_on_the_lanes(n_many, n_few, na):
    rng = np.random.default_rng(3)
    a = np.zeros((na, 4), np.float32)
    a[:, :2] = rng.uniform(-8, 8, (na, 2))
    a[:, 2] = rng.uniform(-1, 0, na)
    a[:, 3] = rng.uniform(-.3, .3, na)
    c = np.stack([rng.uniform(3, 4, na), rng.uniform(.002, .01, na), np.full(na, -1.8), np.zeros(na)], 1)
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v, np.float32), device=dev())    # noqa: E731
    pts = t(D.scan_points([-8, -8, 8], [16 / n_many, 0, 0], [0, 16 / n_many, 0], n_many, n_many))

    def scan(n):
        return D.relax_direct_morse(t(a), t(c), pts[:n], 5, D.Tip(), [0, -.1, .1, 0], [0, 1.8, 0., 0], 40, 1e-8)
    n = n_few * n_few
    for many, few in zip(scan(n_many * n_many), scan(n)):
        assert torch.isfinite(many).all() and torch.equal(many[:n], few)


@pytest.mark.parametrize("lanes", [1, 2, 4])
def test_probe_within_1e_10_of_the_anchor(lanes):
    """A probe that its first step takes to 2^-35 A (3e-11) from the anchor: the spring's length is 1e-10 there, in the
    short forms as in IEEE's.  dt = 1/2 and a constant force of 4 (2^-35 - 2^-28) from the rest position 2^-28, where
    the radial spring is at rest."""
    n = (8, 8, 8)
    sp = D.axis_aligned_spec([-2, -2, -2], [4, 4, 4], n)
    g = np.zeros(n + (4,), np.float32)
    g[..., 0] = 4 * (2.0 ** -35 - 2.0 ** -28)
    tip = D.Tip(stiffness=np.array([0, 0, 0, -1], np.float32), dpos0=np.array([2.0 ** -28, 0, 0, 2.0 ** -28], np.float32),
                relax=np.array([0.5, 0.1, 0.05, 0.5], np.float32), tipC=np.array([0, 0, 1, -0.125], np.float32))
    pts = np.zeros((5, 4), np.float32)
    G, P = (torch.as_tensor(v, device=dev()) for v in (g, pts))
    for cb in (True, False):
        FEs, PPs = D.relax_tilted(G, sp, P, 3, tip, 4, 1e-30, check_before=cb, lanes=lanes)
        FEo, PPo = O.relax_tilted(g, sp.n, sp.dinvA, sp.dinvB, sp.dinvC, pts, 3, tip.tipA, tip.tipB, tip.tipC,
                                  tip.stiffness, tip.dpos0, tip.relax, tip.surfFF, 4, 1e-30, cb, "f32")
        np.testing.assert_array_equal(PPs.cpu().numpy(), PPo)
        np.testing.assert_array_equal(FEs.cpu().numpy(), FEo)
