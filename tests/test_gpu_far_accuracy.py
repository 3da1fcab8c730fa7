"""Accuracy of the interpolated grid projection where its sums differ most from the direct sum's: FP64 sums, fine
grids, steep exponents."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import oracle as O                                     # noqa: E402
from spammm_amd import device as D                                 # noqa: E402
from tests.test_gpu_grid_far import CASES, project, setup, voxel_points      # noqa: E402


@pytest.mark.parametrize("name", ["one_level_morse", "two_levels"])
def test_fp64_sums_do_not_depend_on_the_order_of_the_atoms(name):
    """acc64 adds FP32 terms, the same at any place in the list, in FP64: another order of the atoms moves a sum by
    2^-53 of its terms each, 1e-12 of the sum even where the terms cancel to 1e-2, so the rounded voxels have the same
    bits but for one in 1e4 that lies on the edge of a rounding, and those are neighbours."""
    s = setup(*next(c for c in CASES if c[0] == name)[1:])
    order = np.random.default_rng(3).permutation(len(s[0]))
    a = project(s, acc64=True, cap=False)
    b = project((np.ascontiguousarray(s[0][order]), np.ascontiguousarray(s[1][order])) + s[2:], acc64=True, cap=False)
    off = a != b
    print(f"[acc64] {name}: {int(off.sum())} of {off.numel()} differ")
    assert off.float().mean() <= 1e-3
    assert (((a - b).abs() <= 2.0 ** -23 * a.abs() + 1e-12) | ~off).all()


def heights(s, lo, hi, rng, k):
    """k voxels (indices, flat and by axis) between lo and hi above the grid's z = 0."""
    sp = s[2]
    z = np.arange(sp.n[2]) * sp.dC[2] + sp.p0[2]
    ok = np.nonzero((z >= lo) & (z < hi))[0]
    i = np.stack([rng.integers(0, sp.n[0], k), rng.integers(0, sp.n[1], k), rng.choice(ok, k)], 1)
    return (i[:, 2] * sp.n[1] + i[:, 1]) * sp.n[0] + i[:, 0], i


def values(model, s, i, cp):
    """FP64 field at voxels i (uncapped) of the pair parameters cp, at the FP32 positions of voxels and images."""
    atoms, _, sp, Qs, QZs, npbc, lvA, lvB = s
    f = np.float32
    im = [(f(x), f(y)) for y in range(-npbc[1], npbc[1] + 1) for x in range(-npbc[0], npbc[0] + 1)]
    sites = np.concatenate([np.c_[(atoms[:, :3] + x * lvA) + y * lvB, atoms[:, 3:]] for x, y in im]).astype(f)
    return O.pair_fe(model, sites, np.tile(cp, (len(im), 1)), voxel_points(sp, i), Qs, QZs)


@pytest.mark.parametrize("step,n", [(0.03, (260, 250, 200)), (0.04, (230, 220, 170))])
def test_fine_lj_grids_without_charges(step, n):
    """The r^-13 forces of atoms 10 half-widths (2.3 and 3 A) away.  Against FP64 at the FP32 positions, of the sum of
    the repulsive and attractive fields: differences of positions below 8 A carry 2.4e-7 A, which enter 14 / r-fold
    (1.2e-6 at 2.8 A), a reciprocal root of 1 ulp 14-fold (1.7e-6), the other roundings and the interpolation (kTol)
    1e-6: 5e-6."""
    s = setup(0, 60, 1, n, step, "none", 0.0)[:-2] + tuple(22.0 * np.eye(3, dtype=np.float32)[:2])
    flat, i = heights(s, 2.2, 4.0, np.random.default_rng(2), 20000)
    got = project(s, cap=False).cpu().numpy().reshape(-1, 4)[flat].astype(np.float64)
    one = [values(0, s, i, (s[1] * np.array(m, np.float32))) for m in ((1, 0), (0, 1))]
    err = np.abs(got - (one[0] + one[1])).max(1) / sum(np.linalg.norm(v, axis=1) for v in one)
    print(f"[fine] {step}: largest {err.max():.1e}, rms {np.sqrt((err ** 2).mean()):.1e}")
    assert err.max() <= 5e-6


@pytest.mark.parametrize("step,n,K,tip,charged,lo,hi", [
    (0.2, (110, 110, 110), -1.8, "none", True, 12.0, 19.0),        # above the near radius of every atom
    (0.125, (176, 176, 140), -1.8, "q0", False, 9.0, 15.0),        # a charged tip over atoms without charges
    (0.04, (230, 220, 170), -2.5, "none", True, 2.5, 4.5),
    (0.04, (230, 220, 170), -3.5, "q0", True, 2.5, 4.5),
    (0.1, (130, 130, 120), -1.8, "offsets", True, 3.0, 10.0),      # charges of both signs, interpolated
])
def test_morse_exponents(step, n, K, tip, charged, lo, hi):
    """Against FP64 at the FP32 positions, of the Morse field and (4e-6) of the charge terms: r carries 3 ulp at most, the
    exponent K r 1.5e-5 up to K r = 45, the exponent's rounding 2.6e-6, the rest 1e-6: 2e-5."""
    s = list(setup(1, 60, 1, n, step, tip, 0.0)[:-2] + tuple(22.0 * np.eye(3, dtype=np.float32)[:2]))
    s[1][:, 2] = K
    if not charged:
        s[0][:, 3] = 0.0
    flat, i = heights(s, lo, hi, np.random.default_rng(2), 6000)
    got = project(tuple(s), cap=False).cpu().numpy().reshape(-1, 4)[flat].astype(np.float64)
    want = values(1, s, i, s[1])
    morse = np.linalg.norm(values(1, s[:3] + [[0] * 4] + s[4:], i, s[1]), axis=1)
    P = voxel_points(s[2], i).astype(np.float64)
    S = sum(O.abs_term_sums(s[0], np.zeros((60, 2)), q, s[5], s[6], s[7], P + [0, 0, z]) for q, z in zip(*s[3:5]) if q)
    ratio = np.abs(got - want).max(1) / (2e-5 * morse + 4e-6 * S)
    print(f"[morse] {step} {K} {tip}: largest error / bound {ratio.max():.2e}")
    assert ratio.max() <= 1


def test_time_of_one_level_grows_with_the_sites():
    """Four times the sites take four times as long (and up to 1.4 times that), not sixteen."""
    def ms(na):
        s = list(setup(1, 8, 1, (96, 96, 48), 0.1, "q0", 0.0))
        rng = np.random.default_rng(1)
        s[0], s[1] = (np.repeat(v, na // 8, 0) for v in s[:2])
        s[0][:, :2] = rng.uniform(-50, 50, (na, 2))
        s[-2:] = 100.0 * np.eye(3, dtype=np.float32)[:2]
        project(s)
        t = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        for e in t:
            e.record()
            project(s)
        torch.cuda.synchronize()
        return min(p.elapsed_time(q) for p, q in zip(t, t[1:]))
    few, many = ms(4000), ms(16000)
    print(f"[sites] 36,000 {few:.2f} ms, 144,000 {many:.2f} ms")
    assert many <= 5.6 * few


def gradient(model, atoms, cp, spec, Qs, QZs, cot, lv):
    """d(sum of cot . (F, E)) / d(x, y, z, q, c6 or R0, c12 or E0) of 3 x 3 images in FP64, at the voxels' exact positions."""
    k = (cot != 0).any(-1).nonzero()
    ax = [torch.as_tensor(np.asarray(v, np.float64)[:3], device=cot.device) for v in (spec.p0, spec.dA, spec.dB, spec.dC)]
    P = ax[0] + k[:, 2:] * ax[1] + k[:, 1:2] * ax[2] + k[:, :1] * ax[3]
    g = cot[k[:, 0], k[:, 1], k[:, 2]].double()
    f = np.float32
    charges = [(float(f(q) * f(14.3996448915)), float(f(z))) for q, z in zip(Qs, QZs) if q]     # FP32 in the kernels too
    out = []
    for j in range(len(atoms)):
        v = torch.cat([atoms[j], cp[j]]).double().requires_grad_(True)
        tot = torch.zeros_like(v)
        for iy, ix in np.ndindex(3, 3):
            d = P - v[:3] - torch.as_tensor((ix - 1.0) * lv[0] + (iy - 1.0) * lv[1], device=cot.device).double()
            i2 = 1 / ((d * d).sum(1) + 1e-4)
            gd = (g[:, :3] * d).sum(1)
            if model == 0:
                L = ((v[5] * i2 ** 3 - v[4]) * i2 ** 3 * g[:, 3] + (12 * v[5] * i2 ** 3 - 6 * v[4]) * i2 ** 4 * gd).sum()
            else:
                ex = torch.exp(v[6] * (i2 ** -0.5 - v[4]))
                L = (v[5] * ex * ((ex - 2) * g[:, 3] - 2 * v[6] * (ex - 1) * i2.sqrt() * gd)).sum()
            for q, zo in charges:
                i1 = (d[:, 0] ** 2 + d[:, 1] ** 2 + (d[:, 2] + zo) ** 2 + 1e-4).rsqrt()
                L = L + (q * v[3] * i1 * (g[:, 3] + i1 * i1 * (gd + zo * g[:, 2]))).sum()
            tot += torch.autograd.grad(L, v)[0]
        out.append(tot)
    return torch.stack(out)[:, :6]


# law, step, planes in z, first plane, height of the first plane over the atoms, tip, exponent, cotangent of one sign
ADJOINTS = [(0, 0.05, 448, 400, 3.0, "q0", 0, True), (0, 0.05, 448, 400, 3.0, "offsets", 0, True),
            (0, 0.03, 448, 64, 2.8, "none", 0, False),              # r^-14 terms at the near radius
            (1, 0.1, 448, 64, 11.0, "none", -3.0, False),           # a field of steep exponentials
            (1, 0.1, 448, 64, 3.0, "q0", -1.8, False)]


@pytest.mark.parametrize("model,step,nz,k0,height,tip,K,one_sign", ADJOINTS)
def test_interpolated_adjoint_is_no_further_off_than_the_direct_one(model, step, nz, k0, height, tip, K, one_sign):
    """At least 507 blocks of voxels at once (interpolated, unless the rule refuses) and layer by layer (169: too few,
    direct).  Per column, rms over the atoms against FP64: the near sites' roundings are the same in both, the rest is to
    be smaller; 1.15 allows for chance in 60 to 180 values, 1.3 in those of a cotangent of both signs, whose sums hold
    fewer of their terms."""
    n = (208, 208, nz)
    atoms, cp, _, Qs, QZs, npbc, _, _ = setup(model, 60, 1, (8, 8, 8), step, tip, 0.0)
    if model == 1:
        cp[:, 2] = K
    L = np.array(n) * step
    spec = D.axis_aligned_spec([-L[0] / 2, -L[1] / 2, atoms[:, 2].max() + height - k0 * step], L, n)
    lv = 22.0 * np.eye(3, dtype=np.float32)[:2]
    A, C = (torch.as_tensor(v, device=D.require_gpu()) for v in (atoms, cp))
    cot = torch.zeros((n[2], n[1], n[0], 4), device=A.device)
    r = np.random.default_rng(8).normal(size=(40, n[1], n[0], 4)).astype(np.float32)
    cot[k0:k0 + 40] = torch.as_tensor(1 + 0.2 * np.abs(r) if one_sign else r)
    grid = torch.zeros_like(cot)
    params = model == 0

    def grad(c):
        return D.grid_adjoint(A, C, model, spec, Qs, QZs, grid, c, npbc, *lv, cap=True, params=params).to(A.device)
    whole, direct = grad(cot), 0
    for k in range(k0, k0 + 40, 16):
        part = torch.zeros_like(cot)
        part[k:k + 16] = cot[k:k + 16]
        direct = direct + grad(part)
    want = gradient(model, A, C, spec, Qs, QZs, cot, lv)
    cols = [slice(0, 3)] + [3] * (tip != "none") + [4, 5] * params
    rms = [[float((g - want)[:, c].square().mean().sqrt()) for c in cols] for g in (whole, direct)]
    print(f"[adjoint] {model} {step} {tip} {K}: rms error interpolated / direct of columns:",
          *(f"{a / b:.2f}" for a, b in zip(*rms)))
    assert all(a <= (1.15 if one_sign else 1.3) * b for a, b in zip(*rms))
