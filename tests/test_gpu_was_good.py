"""A frame's refPixelWasGood mask begins with its first evaluation at level 1:
an alignment that fails before (no depth to align to, or too few points at a
coarse level) leaves a frame without one, and createKeyFrame then tests the
residuals of the pixels it propagates instead of the mask."""
import numpy as np
import pytest

import lsdg
import synth

pytestmark = pytest.mark.gpu


def _fail(ctx, how, cam, img, kf, frame):
    if how == "no depth":
        bare = ctx.frame(7, cam, img)
        ref = ctx.ref(bare)
        with pytest.raises(lsdg.LsdgError):
            ctx.se3_track(ref, frame, synth.IDENTITY7)
        ref.destroy()
        bare.destroy()
    elif how == "few points":
        p = lsdg.default_params()
        p.min_goodperall_pixel_absmin = 2.0  # more points than the coarsest level has
        ctx.set_params(p)
        ref = ctx.ref(kf)
        try:
            _, st, status = ctx.se3_track(ref, frame, synth.IDENTITY7)
        finally:
            ctx.set_params(lsdg.default_params())
        assert status == lsdg.DIVERGED and st.num_residual_calls[1] == 0
        ref.destroy()


@pytest.mark.parametrize("how", ["no depth", "few points"])
def test_failed_alignment_leaves_no_mask(ctx, how):
    cam = synth.camera(200, 152)
    rng = np.random.default_rng(3)
    img = rng.integers(0, 256, (152, 200)).astype(np.uint8)
    other = rng.integers(0, 256, (152, 200)).astype(np.uint8)  # residuals that the test refuses
    idepth = rng.uniform(0.9, 1.1, img.shape).astype(np.float32)
    var = np.full(img.shape, 0.01, np.float32)
    ones = np.ones((76, 100), np.uint8)
    maps = []
    for mask, fail in ((None, None), (None, how), (ones, None)):
        kf, nkf = ctx.frame(0, cam, img), ctx.frame(1, cam, other)
        kf.set_depth(idepth, var)
        nkf.set_tracking(kf, [0, 0, 0, 1, 0.01, 0.0, 0.0, 1], 0.3, mask)
        if fail:
            _fail(ctx, fail, cam, img, kf, nkf)
        dm = ctx.depthmap(cam)
        dm.set_prior(kf, idepth, var, 30)
        dm.create_keyframe(nkf)
        maps.append(dm.read())
        for x in (dm, nkf, kf):
            x.destroy()
    plain, failed, masked = maps
    # the two rules keep different pixels here, so a stray mask shows
    assert plain["is_valid"].any() and not np.array_equal(plain["is_valid"], masked["is_valid"])
    for k in plain:
        assert np.array_equal(plain[k].view(np.uint8), failed[k].view(np.uint8)), k
