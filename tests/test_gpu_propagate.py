"""createKeyFrame's propagation where destinations have many sources: a camera
that steps back gathers up to hundreds of old pixels in one new one, and they
fold in raster order whatever order the device listed them in.  Two
propagations in a row (the second finds the lists empty again), every field
bit-exact against the restatement with FP64 accumulation, at a ragged size."""
import numpy as np
import pytest

import lsdg
import pyoracle
import synth

pytestmark = pytest.mark.gpu

FIELDS = ["is_valid", "blacklisted", "next_stereo_frame_min_id", "validity_counter", "idepth", "idepth_var",
          "idepth_smoothed", "idepth_var_smoothed"]


def _run(sys_, cam, img, idepth, var, back):
    im = img.astype(np.float32)
    kf = sys_.frame(0, cam, im)
    k2, k3 = sys_.frame(1, cam, im), sys_.frame(2, cam, im)
    ones = np.ones((cam["h"] >> 1, cam["w"] >> 1), np.uint8)
    k2.set_tracking(kf, [0, 0, 0, 1, 0.01, 0.0, -back, 1], 0.3, ones)
    k3.set_tracking(k2, [0, 0, 0, 1, 0.0, 0.005, 0.0, 1], 0.3, ones)
    dm = sys_.depthmap(cam)
    dm.set_prior(kf, idepth, var, 30)
    out = []
    for k in (k2, k3):
        dm.create_keyframe(k)
        out.append((dm.read(), k.get_tracking()[1], [k.read(lsdg.WHAT_IDEPTH, l) for l in range(5)],
                    [k.read(lsdg.WHAT_IDEPTH_VAR, l) for l in range(5)]))
    return out


# sources per destination: 1 (no step back), about 4, about 36, about 300
@pytest.mark.parametrize("back", [0.0, 2.0, 10.0, 35.0])
def test_many_sources_per_destination(ctx, back):
    cam = synth.camera(202, 138)
    rng = np.random.default_rng(8)
    img = rng.integers(0, 256, (138, 202)).astype(np.uint8)  # strong gradients everywhere
    idepth = rng.uniform(0.45, 0.55, img.shape).astype(np.float32)
    var = rng.uniform(0.001, 0.02, img.shape).astype(np.float32)
    p = pyoracle.default_params()
    p.min_abs_grad_decrease = 0.0
    ctx.set_params(p)
    try:
        g = _run(ctx, cam, img, idepth, var, back)
    finally:
        ctx.set_params(lsdg.default_params())
    o = _run(pyoracle.Oracle(2, params=p), cam, img, idepth, var, back)
    for (gh, gt, gd, gv), (oh, ot, od, ov) in zip(g, o):
        assert gh["is_valid"].any()
        for k in FIELDS:
            assert np.array_equal(gh[k].view(np.uint8), oh[k].view(np.uint8)), k
        assert np.array_equal(gt, ot)
        for a, b in zip(gd + gv, od + ov):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
