"""Single evaluations over counts of points with one block, two, a few, the
most, and the most with several points per thread: block 0's merge of the
others' rows against the oracle's sums of the same FP32 terms."""
import numpy as np
import pytest

import lsdg
import pyoracle
import synth

pytestmark = pytest.mark.gpu

MOST = 128 * 256  # points that one pass of the largest grid takes


@pytest.mark.parametrize("n", [1, 256, 257, 3 * 256 + 1, 4 * 256, 5 * 256, 37 * 256 + 5, MOST, MOST + 1, 2 * MOST + 77])
def test_rows_of_every_block_are_added(ctx, n):
    cam = synth.camera(640, 480)
    d = synth.sim3_instance(71, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
    # one pixel with depth for each of n interior pixels of level 1
    at = np.random.default_rng(n).permutation(318 * 238)[:n]
    y, x = 2 * (at // 318 + 1), 2 * (at % 318 + 1)
    idepth, var = np.full((480, 640), -1, np.float32), np.full((480, 640), -1, np.float32)
    idepth[y, x], var[y, x] = 0.5 + 0.3 * np.sin(0.01 * x), 0.01
    pose = [*synth.sample_pose(77, 0.01, 0.5), 1.02]
    res = []
    for c in (ctx, pyoracle.Oracle(2)):
        a = c.frame(0, cam, d["a_img"].astype(np.float32))
        a.set_depth(idepth, var)
        b = c.frame(1, cam, d["b_img"].astype(np.float32))
        b.set_depth(d["b_idepth"], d["b_var"])
        ref = c.ref(a)
        res.append([c.se3_evaluate(ref, b, 1, pose[:7])[0], c.sim3_evaluate(ref, b, 1, pose)])
    for u, v in zip(*res):
        assert u.warped_count == v.warped_count > 0.8 * n - 1
        # FP64 sums of at most n equal FP32 terms, in another order: n 2^-53 of their magnitudes
        for p, q in ((np.array(u.A[:]), np.array(v.A[:])), (np.array(u.b[:]), np.array(v.b[:]))):
            assert np.abs(p - q).max() <= 1e-12 * np.abs(q).max() + 1e-300
        assert abs(u.error - v.error) <= 1e-12 * abs(v.error) and abs(u.usage - v.usage) <= 1e-12 * v.usage
