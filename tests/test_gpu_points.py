"""Point clouds of several levels at once: every level's points in row-major
order with the pixel's depth, variance and gradient, at sizes around a tile,
without points, with every interior pixel, and past the sizes up to which
storage is taken for every pixel and tiles add up the counts before them
themselves (4228 tiles, and 8409: three rounds of the scan); after a depth change, and when an alignment
builds them before the host knows their counts."""
import numpy as np
import pytest

import lsdg
import synth

pytestmark = pytest.mark.gpu


def _expect(kf, level, img):
    d, v = kf.read(lsdg.WHAT_IDEPTH, level), kf.read(lsdg.WHAT_IDEPTH_VAR, level)
    m = np.zeros(d.shape, bool)
    m[1:-1, 1:-1] = ~((v <= 0) | (d == 0))[1:-1, 1:-1]
    return np.flatnonzero(m), d.ravel()[m.ravel()], v.ravel()[m.ravel()]


@pytest.mark.parametrize("w,h,density", [(64, 64, 0.3), (66, 98, 1.0), (130, 94, 0.0), (642, 482, 0.25),
                                         (2402, 1802, 0.02), (4100, 2100, 0.05)])
def test_levels_are_compacted_in_order(ctx, w, h, density):
    rng = np.random.default_rng(w)
    cam = synth.camera(w, h)
    img = rng.integers(0, 255, (h, w)).astype(np.uint8)
    kf = ctx.frame(0, cam, img)
    fr = ctx.frame(1, cam, img)
    ref = ctx.ref(kf)
    for k in range(2):  # a second depth, with other counts
        keep = rng.random((h, w)) < density * (1 - 0.5 * k)
        d = np.where(keep, rng.uniform(0.3, 2.0, (h, w)), -1).astype(np.float32)
        kf.set_depth(d, np.where(keep, 0.01, -1).astype(np.float32))
        if k == 1:
            ctx.se3_track(ref, fr, synth.IDENTITY7)  # queues levels 1-4 and learns their counts
        for level in (3, 0, 1, 2, 4):
            at, di, va = _expect(kf, level, img)
            p = ref.points(level)
            assert len(p) == len(at) == ref.num_points(level)
            assert np.array_equal(p[:, 7].astype(np.int64), at.astype(np.float32).astype(np.int64))
            assert np.array_equal(p[:, 2], np.float32(1) / di) and np.array_equal(p[:, 4], va)
            I = kf.read(lsdg.WHAT_IMAGE, level)
            g = kf.read(lsdg.WHAT_GRADIENTS, level).reshape(-1, 4)
            assert np.array_equal(p[:, 3], I.ravel()[at])
            assert np.array_equal(p[:, 5], g[at, 0]) and np.array_equal(p[:, 6], g[at, 1])
    for x in (ref, fr, kf):
        x.destroy()
