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


def test_mask_after_alignments_that_wrote_none(ctx):
    """The first alignment that reaches level 1 starts from an all-ones mask,
    however many failed before it."""
    cam = synth.camera(200, 152)
    d = synth.sim3_instance(41, cam=cam, max_trans=0.02, max_rot_deg=0.5, scale_range=(1.0, 1.0))
    kf = ctx.frame(0, cam, d["a_img"])
    kf.set_depth(d["a_idepth"], d["a_var"])
    ref = ctx.ref(kf)
    masks = []
    for failures in ([], ["no depth"], ["few points", "few points"], ["few points", "no depth", "few points"]):
        fr = ctx.frame(1, cam, d["b_img"])
        for how in failures:
            _fail(ctx, how, cam, d["a_img"], kf, fr)
        assert (fr.read(lsdg.WHAT_REF_PIXEL_WAS_GOOD) == 1).all()
        _, _, status = ctx.se3_track(ref, fr, synth.IDENTITY7)
        assert status == lsdg.OK
        masks.append(fr.read(lsdg.WHAT_REF_PIXEL_WAS_GOOD))
        # and a failure afterwards leaves it
        _fail(ctx, "few points", cam, d["a_img"], kf, fr)
        assert np.array_equal(fr.read(lsdg.WHAT_REF_PIXEL_WAS_GOOD), masks[-1])
        fr.destroy()
    assert (masks[0] == 0).any() and all(np.array_equal(m, masks[0]) for m in masks)
    ref.destroy()
    kf.destroy()
