"""Single evaluations over counts of points with one block, two, a few, 128,
128 with several points per thread, and either side of the counts from which
there are 256 and 512: block 0's merge of the others' rows against the oracle's
sums of the same FP32 terms."""
import numpy as np
import pytest

import lsdg
import pyoracle
import synth

pytestmark = pytest.mark.gpu

MOST = 128 * 256  # points that one pass of 128 blocks takes


def _compare(ctx, w, h, level, at, n):
    """Both kinds' evaluation at `level` with depth on the level's interior
    pixels `at` alone."""
    cam = synth.camera(w, h)
    d = synth.sim3_instance(71, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
    iw = (w >> level) - 2
    y, x = (at // iw + 1) << level, (at % iw + 1) << level
    idepth, var = np.full((h, w), -1, np.float32), np.full((h, w), -1, np.float32)
    idepth[y, x], var[y, x] = 0.5 + 0.3 * np.sin(0.01 * x), 0.01
    pose = [*synth.sample_pose(77, 0.01, 0.5), 1.02]
    res = []
    for c in (ctx, pyoracle.Oracle(2)):
        a = c.frame(0, cam, d["a_img"].astype(np.float32))
        a.set_depth(idepth, var)
        b = c.frame(1, cam, d["b_img"].astype(np.float32))
        b.set_depth(d["b_idepth"], d["b_var"])
        ref = c.ref(a)
        assert ref.num_points(level) == n
        res.append([c.se3_evaluate(ref, b, level, pose[:7])[0], c.sim3_evaluate(ref, b, level, pose)])
    for u, v in zip(*res):
        assert u.warped_count == v.warped_count > 0.8 * n - 1
        # FP64 sums of at most n equal FP32 terms, in another order: n 2^-53 of their magnitudes
        bound = max(1e-12, n * 2.0 ** -53)
        for p, q in ((np.array(u.A[:]), np.array(v.A[:])), (np.array(u.b[:]), np.array(v.b[:]))):
            assert np.abs(p - q).max() <= bound * np.abs(q).max() + 1e-300
        assert abs(u.error - v.error) <= bound * abs(v.error) and abs(u.usage - v.usage) <= bound * v.usage


@pytest.mark.parametrize("n", [1, 256, 257, 3 * 256 + 1, 4 * 256, 5 * 256, 37 * 256 + 5, MOST, MOST + 1, 2 * MOST + 77])
def test_rows_of_every_block_are_added(ctx, n):
    # one pixel with depth for each of n interior pixels of level 1
    _compare(ctx, 640, 480, 1, np.random.default_rng(n).permutation(318 * 238)[:n], n)


@pytest.mark.parametrize("n", [5 * MOST - 1, 5 * MOST, 32 * MOST - 1, 32 * MOST, 32 * MOST + 129])
def test_rows_of_large_grids_are_added(ctx, n):
    _compare(ctx, 1200, 1000, 0, np.random.default_rng(n).permutation(1198 * 998)[:n], n)
