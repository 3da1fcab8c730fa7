"""The batched grid launch at each form of a grid (direct, one level, two levels), model and tip: the stored planes of
every molecule have the plain projection's bits, at both tile sizes and at windows that begin within a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from spammm_amd import _lib, batch as B, device as D, workloads as W      # noqa: E402

TIPS = {"point": ([-0.1, 0, 0, 0], [0, 0, 0, 0]), "pair": ([0, -0.1, 0.1, 0], [0, 1.8, 3.6, 0]), "none": ([0] * 4, [0] * 4)}


@pytest.mark.parametrize("vz", [4, 8])
@pytest.mark.parametrize("tip", TIPS)
@pytest.mark.parametrize("model", [_lib.PPM_MODEL_LJ, _lib.PPM_MODEL_MORSE])
def test_batched_planes_have_the_plain_projections_bits(model, tip, vz):
    mols = []
    for k, (na, n) in enumerate([(7, (50, 45, 40)), (60, (130, 121, 150)), (150, (250, 243, 200))]):
        rng = np.random.default_rng(40 + k)
        w = W.batch_molecule(k)
        w.enames, pos = W.flake_geometry(na, rng)
        w.atoms = np.zeros((na, 4), np.float32)
        w.atoms[:, :3], w.atoms[:, 3] = pos, rng.uniform(-0.3, 0.3, na)
        w.atoms[::5, 3] = 0
        w.cLJ = W._lj_params(w.enames)
        w.n, w.L = n, (np.array(n) * 0.1).astype(np.float32)
        w.p0 = np.array([-w.L[0] / 2, -w.L[1] / 2, -6.0 - 0.3 * k], np.float32)
        w.nxy, w.nz = (9, 7), 12
        w.scan_p0 = np.array([-1, -1, [0.5, 9.0, 10.0][k]], np.float32)
        w.Qs, w.QZs = (np.array(v, np.float32) for v in TIPS[tip])
        mols.append(w)
    cp = None
    if model == _lib.PPM_MODEL_MORSE:
        cp = [np.c_[np.full(len(w.atoms), 3.5), np.full(len(w.atoms), 0.005), np.full(len(w.atoms), -1.8),
                    np.zeros(len(w.atoms))].astype(np.float32) for w in mols]
    bf = B.BatchForward(mols, model=model, cpars=cp)
    bf.launch(B.LaunchConfig(vz=vz))
    err, _ = bf.status()
    assert err == 0
    assert any(klo % 16 for klo, _ in bf.windows)
    for i, (w, sp, d, (klo, nzw)) in enumerate(zip(mols, bf.specs, bf.descs_host, bf.windows)):
        a = slice(d.atom_off, d.atom_off + d.na)
        G = D.grid_project(bf.atoms[a].contiguous(), bf.cpar[a].contiguous(), model, sp, bf.Qs, bf.QZs, w.npbc, w.lvA,
                           w.lvB, cap=bf.cap)[klo:klo + nzw]
        got = bf.grids.view(-1, 4)[d.grid_off:d.grid_off + nzw * d.nx * d.ny].view(G.shape)
        assert torch.equal(got, G), f"molecule {i}, planes {klo}..{klo + nzw}"
