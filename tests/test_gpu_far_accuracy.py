"""Accuracy of the interpolated grid projection where its sums differ most from the direct sum's: FP64 sums, fine
grids, steep exponents."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tests.test_gpu_grid_far import CASES, project, setup      # noqa: E402


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
