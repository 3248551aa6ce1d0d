"""Objects made in memory that earlier objects of the context gave back: they
read nothing of what those left there, whatever the order of sizes, kinds and
destruction, and a batch that runs once gives what a kept plan gives."""
import queue
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


def test_another_thread_destroys_while_the_owner_creates(ctx):
    """Frames and references of one context, given back by a second thread
    while the owner makes the next ones in their memory: none is handed out
    while the other still holds it."""
    cam = synth.camera(160, 120)
    rng = np.random.default_rng(9)
    images = [rng.integers(0, 256, (120, 160)).astype(np.uint8) for _ in range(4)]
    depth, var = np.full((120, 160), 1.0, np.float32), np.full((120, 160), 0.01, np.float32)
    q = queue.Queue()
    errors = []

    def destroy():
        try:
            for x in iter(q.get, None):
                x.destroy()
        except Exception as e:  # reported below
            errors.append(e)

    t = threading.Thread(target=destroy)
    t.start()
    held = []
    try:
        for k in range(200):
            f = ctx.frame(k, cam, images[k % 4])
            f.set_depth(depth, var)
            r = ctx.ref(f)
            n = r.num_points(1)
            held.append((k, f, r, n))
            if len(held) > 3:
                j, f, r, n = held.pop(0)
                assert np.array_equal(f.read(lsdg.WHAT_IMAGE, 0), images[j % 4].astype(np.float32))
                p = r.points(1)
                assert len(p) == n and (p[:, 2] == 1.0).all()
                q.put(r)
                q.put(f)
        for _, f, r, _ in held:
            q.put(r)
            q.put(f)
    finally:
        q.put(None)
        t.join()
    assert not errors
