"""The epipolar search over 8-bit images in their packed form: the same map,
bit for bit, as over float images of the same values, whichever way the 8-bit
image came in, with references in the kernel arguments and in memory, at sizes
that end inside a tile; mixed updates take the float form."""
import numpy as np
import pytest

import lsdg
import synth

pytestmark = pytest.mark.gpu


def _identity_table(cam):
    y, x = np.mgrid[0:cam["h"], 0:cam["w"]].astype(np.float32)
    # the last row and column have no second tap: no source
    ok = (x < cam["w"] - 1) & (y < cam["h"] - 1)
    return np.stack([np.where(ok, x, -1), np.where(ok, y, -1)], -1).astype(np.float32)


def _run(ctx, cam, imgs, poses, seed, make):
    frames = [make(k, im) for k, im in enumerate(imgs)]
    kf = frames[0]
    for f, p in zip(frames[1:], poses[1:]):
        f.set_tracking(kf, [*p, 1.0], 0.4)
    dm = ctx.depthmap(cam)
    dm.init_random(kf, seed)
    dm.update([frames[1]])
    dm.update(frames[2:4])
    dm.update(frames[1:])  # more references than ride in the kernel arguments
    out = dm.read()
    for x in [dm, *frames]:
        x.destroy()
    return out


@pytest.mark.parametrize("w,h", [(64, 64), (202, 138), (322, 242)])
def test_packed_equals_float(ctx, w, h):
    cam = synth.camera(w, h)
    sc = synth.Scene(17)
    poses = [np.array([*synth.sample_pose(60 + k, 0.0, 0.3)[:4], 0.02 * k, 0.004 * k, 0.002 * k]) for k in range(7)]
    poses[0] = np.array(synth.IDENTITY7)
    und = ctx.undistorter((w, h), _identity_table(cam))
    imgs = []
    for k, p in enumerate(poses):
        im = sc.render(p, cam, 1.0, 90 + k)[0]
        im[-1, :] = im[:, -1] = 0  # what the undistorter leaves there
        imgs.append(im)

    def ingested(k, im):
        f = ctx.frame(k, cam, np.zeros_like(im))
        f.ingest(k, und, im)
        return f

    makers = [lambda k, im: ctx.frame(k, cam, im.astype(np.float32)), lambda k, im: ctx.frame(k, cam, im), ingested,
              lambda k, im: ctx.frame(k, cam, im if k % 2 else im.astype(np.float32))]
    res = [_run(ctx, cam, imgs, poses, 5, m) for m in makers]
    assert (res[0]["observe_code"] == lsdg.OBS["UPDATED"]).sum() > 20
    for r in res[1:]:
        for k in res[0]:
            assert np.array_equal(r[k].view(np.uint8), res[0][k].view(np.uint8)), k
    und.close()


def test_new_images_keep_their_pixels(ctx):
    """Level 0 and the packed form come from one launch over 2x2 blocks: level
    0 equals the input at sizes with partial tiles and with row padding."""
    rng = np.random.default_rng(3)
    for w, h in [(64, 64), (66, 98), (130, 94), (258, 34 * 2)]:
        im = rng.integers(0, 256, (h, w)).astype(np.uint8)
        f = ctx.frame(0, synth.camera(w, h), im)
        assert np.array_equal(f.read(lsdg.WHAT_IMAGE, 0), im.astype(np.float32))
        a = im.astype(np.float32)
        assert np.array_equal(f.read(lsdg.WHAT_IMAGE, 1),
                              (a[::2, ::2] + a[::2, 1::2] + a[1::2, ::2] + a[1::2, 1::2]) * np.float32(0.25))
        f.destroy()
