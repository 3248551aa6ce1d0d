"""The FP32 evaluation's unscaled divisions (shared correctly rounded
reciprocals) and the scaled ones they fall back to at the ends of the exponent
range: both give the oracle's terms, so the sums agree as in the plain parity
tests wherever the depths' unit puts the denominators.  The operations
themselves are compared with correctly rounded ones over every significand."""
import ctypes as C
import os

import numpy as np
import pytest

import lsdg
import pyoracle
import synth

pytestmark = pytest.mark.gpu

IDENT = np.array([0.0, 0.0, 0.0, 1.0])


def _close(a, b, what):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert np.array_equal(np.isnan(a), np.isnan(b)), what
    # the same FP32 terms, summed in FP64 in another order: 2^-53 per addition
    # of at most a few thousand points, against the largest sum of the kind
    assert np.nanmax(np.abs(a - b)) <= 1e-12 * max(np.nanmax(np.abs(b)), 1e-300), what


# depth unit 2^k: the fast range ends at 2^20; mixed: one point in five at
# 2^22; tiny: a translation whose products fall below the numerators' bound
@pytest.mark.parametrize("k,mixed,trans", [(0, False, 1.0), (18, False, 1.0), (21, False, 1.0), (60, False, 1.0),
                                           (-18, False, 1.0), (-22, False, 1.0), (-30, False, 1.0), (0, True, 1.0),
                                           (0, False, 1e-30), (0, False, 0.0)])
def test_evaluations_at_the_ends_of_the_range(ctx, k, mixed, trans):
    cam = synth.camera(160, 120)
    d = synth.sim3_instance(311, cam=cam, fraction=0.4)
    unit = np.float32(2.0 ** k)
    scale = np.full(d["a_idepth"].shape, 1 / unit, np.float32)
    if mixed:
        scale.ravel()[::5] = np.float32(2.0 ** -22)
    ai = np.where(d["a_idepth"] > 0, d["a_idepth"] * scale, -1).astype(np.float32)
    bi = np.where(d["b_idepth"] > 0, d["b_idepth"] / unit, -1).astype(np.float32)
    rot = synth.sample_pose(5, 0.0, 0.4)[:4]
    pose = [*rot, *(np.array([0.01, -0.004, 0.006]) * float(unit) * trans), 1.01]
    kf = ctx.frame(0, cam, d["a_img"])
    kf.set_depth(ai, d["a_var"])
    fr = ctx.frame(1, cam, d["b_img"])
    fr.set_depth(bi, d["b_var"])
    ref = ctx.ref(kf)
    o = pyoracle.Oracle(2)
    okf = o.frame(0, cam, d["a_img"].astype(np.float32))
    okf.set_depth(ai, d["a_var"])
    ofr = o.frame(1, cam, d["b_img"].astype(np.float32))
    ofr.set_depth(bi, d["b_var"])
    oref = o.ref(okf)
    for level in (1, 2):
        g, _ = ctx.se3_evaluate(ref, fr, level, pose[:7])
        e = o.se3_evaluate(oref, ofr, level, pose[:7])
        e = e[0] if isinstance(e, tuple) else e
        assert g.warped_count == e.warped_count and g.good_count == e.good_count and g.bad_count == e.bad_count
        assert g.warped_count > 100
        s3, q3 = ctx.sim3_evaluate(ref, fr, level, pose), o.sim3_evaluate(oref, ofr, level, pose)
        for a, b, n in ((g, e, "se3"), (s3, q3, "sim3")):
            _close(a.A[:], b.A[:], n)
            _close(a.b[:], b.b[:], n)
            _close([a.error], [b.error], n)
            _close([a.usage], [b.usage], n)
    for x in (ref, fr, kf):
        x.destroy()


@pytest.mark.parametrize("what,least", [("reciprocals", 2 * 121 << 23), ("square roots", 121 << 23),
                                        ("quotients", 50 << 23)])
def test_unscaled_operations_round_correctly(what, least):
    """oracle/rounding_check.hip: reciprocals and square roots of every float
    from 2^-60 to 2^61, quotients for every significand of the denominator."""
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle", "librounding_check.so")
    if not os.path.exists(path):
        pytest.fail(f"{path} is not built; run `make -C oracle`")
    L = C.CDLL(path)
    out, example = (C.c_ulonglong * 2)(), (C.c_uint * 4)()
    assert L.rounding_check(["reciprocals", "square roots", "quotients"].index(what), out, example) == 0
    assert out[1] == 0, [hex(v) for v in example]
    assert out[0] >= least
