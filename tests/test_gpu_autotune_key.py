"""The tuner's cache key names what the timings hold for: the library's build and the batch's kernels."""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


def test_signature_names_the_build_the_model_and_the_tip():
    from spammm_amd import _lib, autotune, batch as B, workloads as W

    def batch(tip=(0.0, 0.0, 0.0, 0.0), **kw):
        mols = [W.batch_molecule(k) for k in range(2)]
        for w in mols:
            w.n, w.nxy = (40, 40, 40), (8, 8)
            w.Qs, w.QZs = np.array([-0.1, 0, 0, 0], np.float32), np.array(tip, np.float32)
        return B.BatchForward(mols, **kw)
    a, b = batch(), batch((1.8, 0, 0, 0))
    c = batch(model=_lib.PPM_MODEL_MORSE, cpars=[np.tile(np.array([3.5, 0.005, -1.8, 0], np.float32),
                                                         (w.atoms.shape[0], 1)) for w in a.molecules])
    keys = [autotune.signature(v) for v in (a, b, c)]
    assert len(set(keys)) == 3
    with open(_lib.LIB_PATH, "rb") as f:
        build = hashlib.sha256(f.read()).hexdigest()[:12]
    assert all(build in k for k in keys)
