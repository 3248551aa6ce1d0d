"""GPU parity of the keyframe export (publishKeyframe's InputPointDense
records and Keyframe::computeVbo's filter, lib/Pangolin_IOWrapper/) against
the oracle's restatement: records and vertices bit-exact, vertex order
included."""
import numpy as np
import pytest

import lsdg
import pyoracle
import synth

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint8)


@pytest.fixture(scope="module")
def keyframes(ctx):
    """The depth workload's keyframe with its true inverse depth on the prior's
    30% of pixels (small variances, so that the filter keeps a good part)."""
    d = synth.depth_instance()
    cam = d["cam"]
    rng = np.random.default_rng(11)
    idp = np.where(d["prior_idepth"] > 0, 1.0 / d["kf_depth"], -1).astype(np.float32)
    var = np.where(idp > 0, rng.uniform(1e-7, 3e-6, idp.shape), -1).astype(np.float32)
    g = ctx.frame(0, cam, d["kf_img"])
    g.set_depth(idp, var)
    o = pyoracle.Oracle(0)
    of = o.frame(0, cam, d["kf_img"].astype(np.float32))
    of.set_depth(idp, var)
    return g, of, o


@pytest.mark.parametrize("level", [0, 1, 3])
def test_keyframe_points_bit_exact(keyframes, level):
    g, of, _ = keyframes
    a, b = g.keyframe_points(level), of.keyframe_points(level)
    assert np.array_equal(_bits(a), _bits(b))
    assert (a["idepth"] > 0).sum() > 100


@pytest.mark.parametrize("level,scale", [(0, 1.0), (0, 30.0), (1, 1.0), (2, 0.5)])
def test_keyframe_vbo_bit_exact(keyframes, level, scale):
    g, of, o = keyframes
    p = lsdg.vbo_params(scale)
    got = g.keyframe_vbo(level, p)
    w, h = of.size(level)
    want = o.compute_vbo(of.keyframe_points(level), w, h, of.camera(level), p)
    assert len(got) == len(want) and len(want) > 50
    assert np.array_equal(_bits(got), _bits(want))


@pytest.mark.parametrize("near", [1, 9])
def test_points_vbo_edge_records(ctx, near):
    """Host records with invalid, NaN, zero-variance and threshold-boundary
    entries, odd sizes."""
    w, h = 37, 29
    rng = np.random.default_rng(5 + near)
    rec = np.zeros(w * h, lsdg.POINT_DENSE_DTYPE)
    ys, xs = np.mgrid[0:h, 0:w]
    idp = (0.8 + 0.002 * xs + 0.001 * ys).astype(np.float32).ravel()  # a slanted plane
    idp[rng.random(w * h) < 0.04] = -1.0
    idp[rng.random(w * h) < 0.02] = 0.0
    idp[rng.random(w * h) < 0.01] = np.nan
    var = rng.choice(np.array([0.0, 1e-6, 1e-5, 1e-4, 2.4e-4, 5e-4, 2e-3], np.float32), w * h)
    rec["idepth"], rec["idepth_var"] = idp, var
    rec["color"] = rng.integers(0, 256, (w * h, 4), dtype=np.uint8)
    cam4 = (300.0, 280.0, 18.0, 14.0)
    p = lsdg.vbo_params(1.7, min_near_support=near)
    got = ctx.points_vbo(rec, w, h, cam4, p)
    want = pyoracle.Oracle(0).compute_vbo(rec, w, h, cam4, p)
    assert len(got) == len(want) and len(want) > 0
    assert np.array_equal(_bits(got), _bits(want))


def test_no_depth_is_an_error(ctx):
    cam = synth.camera(128, 96)
    f = ctx.frame(0, cam, np.zeros((96, 128), np.uint8))
    with pytest.raises(RuntimeError):
        f.keyframe_points(0)


def _host_memory(n, pinned):
    """n bytes of host memory, pinned by the runtime the library is linked to
    or ordinary, and what frees it."""
    if not pinned:
        return np.zeros(n, np.uint8), lambda: None
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip, p = lsdg.C.CDLL(path), lsdg.C.c_void_p()
    assert hip.hipHostMalloc(lsdg.C.byref(p), lsdg.C.c_size_t(n), 0) == 0
    return np.ctypeslib.as_array((lsdg.C.c_uint8 * n).from_address(p.value)), lambda: hip.hipHostFree(p)


@pytest.mark.parametrize("offset", [0, 4, 8, 12, 16, 4100])
def test_vertices_into_the_middle_of_a_pinned_block(keyframes, offset):
    """The buffer begins anywhere in its block, aligned as a vertex is (4
    bytes); what is beside the vertices stays as it was."""
    g, of, o = keyframes
    p = lsdg.vbo_params(1.0)
    w, h = of.size(0)
    want = np.ascontiguousarray(o.compute_vbo(of.keyframe_points(0), w, h, of.camera(0), p)).tobytes()
    out, free = _host_memory(16 * w * h + offset + 64, True)
    out[:] = 0xA5
    n = lsdg.C.c_int32()
    g.ctx.check(g.ctx.L.lsdg_keyframe_vbo(g.h, 0, lsdg.C.byref(p), out.ctypes.data + offset, lsdg.C.byref(n)),
                "lsdg_keyframe_vbo")
    assert out[offset:offset + len(want)].tobytes() == want and 16 * n.value == len(want)
    assert (out[:offset] == 0xA5).all() and (out[offset + len(want):] == 0xA5).all()
    free()


# tiles of 1024 pixels: one, a whole number of them, one pixel into the next
# wave, round and tile, and more than the kernels add up by themselves
@pytest.mark.parametrize("w,h", [(3, 3), (32, 32), (64, 16), (65, 16), (43, 31), (205, 5), (4100, 1030)])
@pytest.mark.parametrize("pinned", [False, True])
def test_points_vbo_tiles(ctx, w, h, pinned):
    rng = np.random.default_rng(w * h)
    rec = np.zeros(w * h, lsdg.POINT_DENSE_DTYPE)
    rec["idepth"] = np.where(rng.random(w * h) < 0.7, rng.uniform(0.5, 2.0, w * h), -1).astype(np.float32)
    rec["idepth_var"] = 1e-6
    rec["color"] = rng.integers(0, 256, (w * h, 4), dtype=np.uint8)
    cam4, p = (300.0, 280.0, 18.0, 14.0), lsdg.vbo_params(1.0, min_near_support=1)
    out, free = _host_memory(16 * w * h, pinned)
    n = lsdg.C.c_int32()
    ctx.check(ctx.L.lsdg_points_vbo(ctx.h, rec.ctypes.data, w, h, *cam4, lsdg.C.byref(p), out.ctypes.data,
                                    lsdg.C.byref(n)), "lsdg_points_vbo")
    want = pyoracle.Oracle(0).compute_vbo(rec, w, h, cam4, p)
    assert n.value == len(want)
    assert out[:16 * n.value].tobytes() == np.ascontiguousarray(want).tobytes()
    free()
