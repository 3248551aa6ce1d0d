"""The default shape of a batch plan: blocks of 512 threads while jobs are few,
of 256 when they are many (either side of the line on 256 CUs), with and without the affine brightness estimate
(whose sums the kernels leave out otherwise).  Every job takes the LM path of
the same alignment run by itself."""
import pytest

import lsdg
import synth
from helpers import twist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,block", [(3, 512), (51, 512), (52, 256), (96, 256)])
@pytest.mark.parametrize("affine", [0, 1])
@pytest.mark.parametrize("kind", [lsdg.JOB_SE3, lsdg.JOB_SIM3])
def test_default_shape_takes_the_single_alignments_path(kind, affine, n, block):
    params = lsdg.default_params()
    params.use_affine_lightning_estimation = affine
    ctx = lsdg.Context(0, params)
    cam = synth.camera(160, 120)
    pairs, jobs, inits = [], [], []
    for k in range(3):
        d = synth.sim3_instance(61 + k, cam=cam, max_trans=0.03, max_rot_deg=1.0, scale_range=(0.98, 1.02))
        a = ctx.frame(2 * k, cam, d["a_img"])
        a.set_depth(d["a_idepth"], d["a_var"])
        b = ctx.frame(2 * k + 1, cam, d["b_img"])
        b.set_depth(d["b_idepth"], d["b_var"])
        pairs.append((ctx.ref(a), b))
    for i in range(n):
        ref, b = pairs[i % 3]
        inits.append([*synth.sample_pose(900 + i // 3, 0.002, 0.1), 1.0])
        jobs.append(lsdg.Job(ref.h, b.h, lsdg.pose8(inits[-1]), kind, 4, 1, 0))
    plan = ctx.batch(jobs)
    assert plan.config()["coop_block"] == block
    res = plan.run()
    for i in list(range(3)) + list(range(n - 3, n)):
        ref, b = pairs[i % 3]
        if kind == lsdg.JOB_SE3:
            pose, st, status = ctx.se3_track(ref, b, inits[i][:7])
            assert res[i].stats.last_good_count == st.last_good_count
        else:
            pose, st, status = ctx.sim3_track(ref, b, inits[i], 4, 1)
            assert abs(res[i].frame_to_ref[7] - pose[7]) <= 1e-9
        # the same FP32 terms, sums and solves in another order of FP64
        assert res[i].status == status and twist(res[i].frame_to_ref[:7], pose[:7]) <= 1e-9, i
        assert list(res[i].stats.num_residual_calls) == list(st.num_residual_calls), i
    plan.destroy()
    ctx.close()
