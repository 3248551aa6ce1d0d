"""Objects made in memory that earlier objects of the context gave back: they
read nothing of what those left there, whatever the order of sizes, kinds and
destruction, and a batch that runs once gives what a kept plan gives."""
import threading

import numpy as np
import pytest

import lsdg
import synth

pytestmark = pytest.mark.gpu


def _work(ctx, cam, seed, prec):
    """One pass over every kind of object: frames, point clouds, a batch, a
    depth map; every result as bytes."""
    d = synth.sim3_instance(seed, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
    u8 = np.clip(d["b_img"], 0, 255).astype(np.uint8)
    a = ctx.frame(0, cam, d["a_img"], prec)
    a.set_depth(d["a_idepth"], d["a_var"])
    b = ctx.frame(1, cam, u8, prec)
    b.set_depth(d["b_idepth"], d["b_var"])
    ref = ctx.ref(a)
    out = [b.read(lsdg.WHAT_GRADIENTS, l) for l in range(5)] + [b.read(lsdg.WHAT_REF_PIXEL_WAS_GOOD)]
    out += [a.read(lsdg.WHAT_IDEPTH, l) for l in range(5)]
    for kind in (lsdg.JOB_SE3, lsdg.JOB_SIM3):
        jobs = [lsdg.Job(ref.h, b.h, lsdg.pose8([*synth.IDENTITY7, 1.0]), kind, 4, 1, 1) for _ in range(3)]
        plan = ctx.batch(jobs)
        kept = bytes(plan.run())
        plan.destroy()
        once = (lsdg.JobResult * len(jobs))()
        ctx.check(ctx.L.lsdg_batch_track(ctx.h, (lsdg.Job * len(jobs))(*jobs), len(jobs), once), "lsdg_batch_track")
        assert bytes(once) == kept
        out.append(np.frombuffer(kept, np.uint8))
    dm = ctx.depthmap(cam)
    dm.init_random(a, seed)
    b.set_tracking(a, [*synth.sample_pose(seed, 0.01, 0.2), 1.0], 0.4)
    dm.update([b])
    out += [a.read(lsdg.WHAT_IDEPTH, 0), a.read(lsdg.WHAT_IDEPTH_VAR, 3)]
    for x in (ref, b, dm, a) if seed % 2 else (dm, a, ref, b):
        x.destroy()
    return b"".join(np.ascontiguousarray(o).tobytes() for o in out)


# sizes that reuse each other's blocks, exactly, with room to spare, or not at all
CASES = [(160, 120, 1, lsdg.FP32), (160, 120, 2, lsdg.FP16), (150, 112, 3, lsdg.FP16), (322, 242, 4, lsdg.FP32),
         (160, 120, 5, lsdg.BF16), (320, 240, 6, lsdg.FP32), (64, 64, 7, lsdg.FP32), (322, 242, 8, lsdg.FP16)]


def test_reused_memory_changes_nothing():
    fresh = {}
    for w, h, seed, prec in CASES:
        ctx = lsdg.Context(0)
        fresh[w, h, seed, prec] = _work(ctx, synth.camera(w, h), seed, prec)
        ctx.close()
    bad = []

    def reuse(order):
        ctx = lsdg.Context(0)
        for i in order:
            w, h, seed, prec = CASES[i]
            if _work(ctx, synth.camera(w, h), seed, prec) != fresh[CASES[i]]:
                bad.append(CASES[i])
        ctx.close()

    threads = [threading.Thread(target=reuse, args=(np.random.default_rng(k).permutation(2 * len(CASES)) % len(CASES),))
               for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
