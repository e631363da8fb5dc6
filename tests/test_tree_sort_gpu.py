"""The tree's sort: digit widths from 3 to 8 bits in one to three passes, sizes
at the edges of its tiles (64 items per step, 2,048 per workgroup)."""
import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("n", [1, 2, 64, 65, 2048, 2049, 70001])
def test_points_are_stably_sorted_by_cell(n, level):
    print("tree sort", n, level, flush=True)
    pts = np.random.default_rng(n + level).uniform(0, 1, (n, 3)) ** 2  # uneven cells
    ev = pa.make_fmm_evaluator(pa.Biharmonic3D(), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig("mixed", 3, level, "fmm"))
    ev.set_source_points(pts)
    ev.set_weights(np.ones(n))
    ev.set_target_points(pts[::-1].copy())
    ev.evaluate()
    for which, p in ((0, pts), (1, pts[::-1])):
        info = ev.tree_info(which)
        codes, perm, _, _ = ev.export_tree(which)
        np.testing.assert_array_equal(np.sort(perm), np.arange(n))
        c = codes.astype(np.int64)
        step = np.diff(c)
        assert np.all(step >= 0)
        assert np.all(np.diff(perm)[step == 0] > 0)  # stable
        # The codes are those of the cells that the points lie in: bit k of x, y
        # and z in bits 3 k + 2, 3 k + 1 and 3 k.
        cell = np.clip(np.floor((p[perm] - info["lo"]) * info["inv_cell"]), 0, 2 ** level - 1).astype(np.int64)
        want = sum(((cell[:, a] >> k) & 1) << (3 * k + 2 - a) for a in range(3) for k in range(level))
        np.testing.assert_array_equal(c, want)
