"""The one-launch alignments: the same LM path as the launch-per-evaluation
form they fall back to when their blocks cannot all run at once, over sizes
with one block, a few and the most, and interleaved on several contexts."""
import threading

import numpy as np
import pytest

import lsdg
import pyoracle
import synth
from helpers import twist

pytestmark = pytest.mark.gpu


def _steps_context(monkeypatch):
    """A context whose one-launch alignments give up at the first wait."""
    monkeypatch.setenv("LSDG_TRACK_SPIN_MAX", "0")
    try:
        return lsdg.Context(0)
    finally:
        monkeypatch.delenv("LSDG_TRACK_SPIN_MAX")


def _pair(ctx, cam, seed, prec):
    d = synth.sim3_instance(seed, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
    a = ctx.frame(0, cam, d["a_img"], prec)
    a.set_depth(d["a_idepth"], d["a_var"])
    b = ctx.frame(1, cam, d["b_img"], prec)
    b.set_depth(d["b_idepth"], d["b_var"])
    return a, b, ctx.ref(a)


def _launches(c, align):
    """align()'s result and the launches it took: one of the one-launch form,
    one per evaluation otherwise."""
    c.profile(True)
    try:
        out = align()
        return out, c.kernel_stats(lsdg.KERNEL_EVAL)["launches"]
    finally:
        c.profile(False)


def _fields(st):
    return [st.last_good_count, st.last_bad_count, st.diverged, st.tracking_was_good, *st.num_residual_calls,
            *st.num_warp_update_calls]


# 64x64: every level is small; 130x98: the split threshold; 322x242: ragged; 1282x962: 64 blocks
@pytest.mark.parametrize("w,h", [(64, 64), (130, 98), (322, 242), (1282, 962)])
@pytest.mark.parametrize("prec", [lsdg.FP32, lsdg.FP16])
def test_one_launch_equals_launch_per_evaluation(ctx, monkeypatch, w, h, prec):
    cam = synth.camera(w, h)
    other = _steps_context(monkeypatch)
    for seed in (41, 42):
        res = []
        for c in (ctx, other):
            a, b, ref = _pair(c, cam, seed, prec)
            (p, st, status), n = _launches(c, lambda: c.se3_track(ref, b, synth.IDENTITY7))
            mask = b.read(lsdg.WHAT_REF_PIXEL_WAS_GOOD)
            (q, st3, status3), n3 = _launches(c, lambda: c.sim3_track(ref, b, [*synth.IDENTITY7, 1.0], 4, 1))
            # the form that ran: at 64x64 no level is split, so nothing waits;
            # elsewhere the other context's first alignment gives up, and the
            # ones after it go launch by launch without a try
            if c is ctx or w == 64:
                assert n == 1 and n3 == 1
            else:
                assert n == sum(st.num_residual_calls) + (1 if seed == 41 else 0)
                assert n3 - sum(st3.num_residual_calls) in (0, 1)  # 1: the evaluation for the information matrix
            res.append((p, st, status, mask, q, st3, status3))
            for x in (ref, b, a):
                x.destroy()
        (p, st, status, mask, q, st3, status3), (p2, st2, status2, mask2, q2, st32, status32) = res
        assert status == status2 and status3 == status32
        assert _fields(st) == _fields(st2) and _fields(st3) == _fields(st32)
        # FP64 sums and solves in another order: the FP32 path's terms are the
        # same, so poses agree to the tests' usual 1e-9
        assert twist(p, p2) <= 1e-9 and twist(q[:7], q2[:7]) <= 1e-9 and abs(q[7] - q2[7]) <= 1e-9
        assert np.array_equal(mask, mask2)
        for k in ("last_residual", "last_mean_res", "point_usage", "last_depth_residual", "last_photometric_residual"):
            for u, v in ((st, st2), (st3, st32)):
                assert np.isclose(getattr(u, k), getattr(v, k), rtol=1e-6, equal_nan=True), k
        H, H2 = np.array(st3.hessian[:]), np.array(st32.hessian[:])
        assert np.abs(H - H2).max() <= 1e-9 * max(np.abs(H2).max(), 1e-30)
    other.close()


@pytest.mark.parametrize("prec", [lsdg.FP32, lsdg.BF16])
def test_large_finest_level(ctx, monkeypatch, prec):
    """Down to a level of more than 1.5 Mpixel, which takes more blocks."""
    cam = synth.camera(1402, 1202)
    p = lsdg.default_params()
    p.se3_min_level = 0
    steps = _steps_context(monkeypatch)
    res = []
    try:
        for c in (ctx, steps):
            c.set_params(p)
            a, b, ref = _pair(c, cam, 41, prec)
            (pose, st, status), n = _launches(c, lambda: c.se3_track(ref, b, synth.IDENTITY7))
            (q, st3, status3), n3 = _launches(c, lambda: c.sim3_track(ref, b, [*synth.IDENTITY7, 1.0], 4, 0))
            assert (n == 1 and n3 == 1) if c is ctx else (n > 2 and n3 > 2)
            res.append((pose, q, _fields(st) + [status], _fields(st3) + [status3]))
            for x in (ref, b, a):
                x.destroy()
    finally:
        ctx.set_params(lsdg.default_params())
        steps.close()
    (pose, q, f, f3), (pose2, q2, g, g3) = res
    assert f == g and f3 == g3
    assert twist(pose, pose2) <= 1e-9 and twist(q[:7], q2[:7]) <= 1e-9 and abs(q[7] - q2[7]) <= 1e-9


@pytest.mark.parametrize("steps", [False, True])
def test_sim3_final_level_without_iterations(ctx, monkeypatch, steps):
    """The final evaluation, at a level that has no iterations, is the last
    one whose point usage counts, in both forms as in the oracle."""
    cam = synth.camera(322, 242)
    p = pyoracle.default_params()
    p.max_its_per_lvl[1] = 0
    p.convergence_eps[2] = 0.0  # level 2 ends on an accepted step, so a final evaluation follows
    c = _steps_context(monkeypatch) if steps else ctx
    c.set_params(p)
    try:
        a, b, ref = _pair(c, cam, 43, lsdg.FP32)
        c.profile(True)
        q, st, status = c.sim3_track(ref, b, [*synth.IDENTITY7, 1.0], 4, 1)
        launches = c.kernel_stats(lsdg.KERNEL_EVAL)["launches"]
    finally:
        c.profile(False)
        c.set_params(lsdg.default_params())
    o = pyoracle.Oracle(2, params=p)
    d = synth.sim3_instance(43, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
    oa, ob = o.frame(0, cam, d["a_img"].astype(np.float32)), o.frame(1, cam, d["b_img"].astype(np.float32))
    oa.set_depth(d["a_idepth"], d["a_var"])
    ob.set_depth(d["b_idepth"], d["b_var"])
    oq, ost, ostatus = o.sim3_track(o.ref(oa), ob, [*synth.IDENTITY7, 1.0], 4, 1)
    assert status == ostatus == lsdg.OK and st.num_residual_calls[1] == 0
    assert launches > 1 if steps else launches == 1  # the form that ran
    assert twist(q[:7], oq[:7]) <= 1e-9 and abs(q[7] - oq[7]) <= 1e-9
    # one FP64 sum of FP32 terms in another order, rounded to float
    assert np.isclose(st.point_usage, ost.point_usage, rtol=2.0 ** -22)
    for x in (ref, b, a):
        x.destroy()
    if steps:
        c.close()


@pytest.mark.parametrize("fail_fac", [2.0, 1.7, 3.1])
def test_damping_after_rejections(ctx, monkeypatch, fail_fac):
    """Steps rejected several times in a row multiply the damping by a power of
    the factor: the same power in the one-launch form, the batch and the host's
    LM step (std::pow), also where the factor's powers round."""
    cam = synth.camera(642, 482)
    p = lsdg.default_params()
    for l in range(5):
        p.lambda_fail_fac[l], p.convergence_eps[l], p.step_size_min[l] = fail_fac, 0.9999, 1e-14
    steps = _steps_context(monkeypatch)
    for c in (ctx, steps):
        c.set_params(p)
    try:
        for seed in range(41, 49):
            out = []
            for c in (ctx, steps):
                a, b, ref = _pair(c, cam, seed, lsdg.FP32)
                pose, st, status = c.se3_track(ref, b, synth.IDENTITY7)
                assert sum(st.num_residual_calls) > sum(st.num_warp_update_calls) + 8  # rejections
                out.append((pose, _fields(st), status))
                if c is ctx:
                    plan = c.batch([lsdg.Job(ref.h, b.h, lsdg.pose8([*synth.IDENTITY7, 1.0]), lsdg.JOB_SE3, 4, 1, 1)])
                    res = plan.run()[0]
                    out.append((np.array(res.frame_to_ref[:7]), _fields(res.stats), res.status))
                    plan.destroy()
                for x in (ref, b, a):
                    x.destroy()
            # the sums' order differs, by FP64 rounding
            assert all(twist(o[0], out[0][0]) <= 1e-12 and o[1:] == out[0][1:] for o in out)
    finally:
        ctx.set_params(lsdg.default_params())
        steps.close()


def test_a_context_that_gave_up_tries_again_after_a_while(monkeypatch):
    cam = synth.camera(130, 98)
    c = _steps_context(monkeypatch)
    a, b, ref = _pair(c, cam, 41, lsdg.FP32)
    vain = []
    for _ in range(203):
        (_, st, _), n = _launches(c, lambda: c.se3_track(ref, b, synth.IDENTITY7))
        vain.append(n - sum(st.num_residual_calls))
    assert vain == [1] + [0] * 100 + [1] + [0] * 100 + [1]
    for x in (ref, b, a):
        x.destroy()
    c.close()


def test_more_evaluations_than_one_launch_makes(ctx):
    """An alignment of 70001 evaluations (heavily damped steps towards a smooth
    minimum), where a launch ends after 65536: it is finished launch by launch,
    not reported as done where it stood."""
    cam = synth.camera(64, 64)
    y, x = np.mgrid[0:64, 0:64].astype(np.float64)
    image = lambda u, v: (128 + 50 * np.sin(u / 7.0) + 50 * np.cos(v / 9.0 + u / 31.0)).astype(np.float32)
    idepth = np.full((64, 64), -1, np.float32)
    idepth[16:48, 16:48] = 1.0  # away from the border: no point enters or leaves the image
    var = np.full((64, 64), 0.01, np.float32)
    p = pyoracle.default_params()
    p.se3_min_level, p.se3_max_level = 1, 2
    p.max_its_per_lvl[1], p.lambda_initial[1], p.lambda_success_fac[1] = 70000, 3e4, 1.0
    p.convergence_eps[1], p.step_size_min[1] = 1.0, 0.0

    def align(c):
        kf, fr = c.frame(0, cam, image(x, y)), c.frame(1, cam, image(x - 4.0, y))
        kf.set_depth(idepth, var)
        return c.se3_track(c.ref(kf), fr, synth.IDENTITY7)

    ctx.set_params(p)
    try:
        pose, st, status = align(ctx)
    finally:
        ctx.set_params(lsdg.default_params())
    opose, ost, ostatus = align(pyoracle.Oracle(2, params=p))
    assert ost.num_residual_calls[1] == 70001
    assert status == ostatus and _fields(st) == _fields(ost)
    assert twist(pose, opose) <= 1e-9 and np.isclose(st.last_residual, ost.last_residual, rtol=1e-6)


def test_contexts_align_at_the_same_time():
    """Six threads, each with its own context, aligning at once: every result
    equals the single-threaded one."""
    cam = synth.camera(640, 480)
    out, errors = {}, []

    def work(k):
        try:
            c = lsdg.Context(0)
            a, b, ref = _pair(c, cam, 50, lsdg.FP32)
            out[k] = [c.se3_track(ref, b, synth.IDENTITY7)[0] for _ in range(20)]
            for x in (ref, b, a):
                x.destroy()
            c.close()
        except Exception as e:  # reported below, in the test's own thread
            errors.append(e)

    work("alone")
    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    want = out["alone"][0]
    assert all(twist(p, want) <= 1e-9 for v in out.values() for p in v)
