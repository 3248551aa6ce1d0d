"""What a frame takes of the device's memory, as the header states it, and a
float frame that is given an 8-bit image later (its packed form is made then)."""
import numpy as np
import pytest

import lsdg
import synth

pytestmark = pytest.mark.gpu


def _free_bytes():
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip, free, total = lsdg.C.CDLL(path), lsdg.C.c_size_t(), lsdg.C.c_size_t()
    assert hip.hipMemGetInfo(lsdg.C.byref(free), lsdg.C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec,u8,per_pixel", [(lsdg.FP32, False, 44), (lsdg.FP32, True, 48), (lsdg.BF16, False, 55),
                                               (lsdg.BF16, True, 59)])
def test_frame_memory(prec, u8, per_pixel):
    c = lsdg.Context(0)
    cam = synth.camera(2048, 1536)
    img = np.zeros((1536, 2048), np.uint8 if u8 else np.float32)
    first = c.frame(0, cam, img, prec)  # what the runtime sets up at first use
    before = _free_bytes()
    frames = [c.frame(k, cam, img, prec) for k in range(4)]
    taken = (before - _free_bytes()) / len(frames) / img.size
    # the runtime may round a block up to 2 MiB: 0.7 bytes a pixel
    assert per_pixel - 2 < taken <= per_pixel + 0.7
    for f in (*frames, first):
        f.destroy()
    c.close()


@pytest.mark.parametrize("prec", [lsdg.FP32, lsdg.FP16])
def test_float_frame_takes_an_8_bit_image(ctx, prec):
    in_size, k, out_size = (230, 171), (150.0, 150.0, 114.5, 85.0), (210, 150)
    ok = (150.0, 150.0, 104.5, 74.5)
    cam = dict(w=210, h=150, fx=ok[0], fy=ok[1], cx=ok[2], cy=ok[3])
    und = ctx.undistorter(in_size, lsdg.fov_undistort_table(k, 0.0, in_size, ok, out_size))
    rng = np.random.default_rng(4)
    src = rng.integers(0, 256, (171, 230)).astype(np.uint8)
    moved = np.roll(src, 3, axis=1)
    maps = []
    for made in ("float", "8 bit"):
        kf = ctx.frame_undistorted(0, cam, und, src, prec)
        if made == "float":
            fr = ctx.frame(9, cam, np.zeros((150, 210), np.float32), prec)
            fr.ingest(1, und, moved)
            fr.ingest(1, und, moved)
        else:
            fr = ctx.frame_undistorted(1, cam, und, moved, prec)
        dm = ctx.depthmap(cam)
        dm.init_random(kf, 5)
        fr.set_tracking(kf, [0, 0, 0, 1, 0.02, 0.0, 0.0, 1], 0.4)
        dm.update([fr])
        maps.append(dm.read())
        for x in (dm, fr, kf):
            x.destroy()
    und.close()
    assert (maps[0]["validity_counter"] > 5).any()
    for key in maps[0]:
        assert np.array_equal(maps[0][key].view(np.uint8), maps[1][key].view(np.uint8)), key
