// C-ABI of the keyframe export: publishKeyframe's point records and the
// viewer's computeVbo filter (lib/Pangolin_IOWrapper/PangolinOutputIOWrapper.cpp:42-97,
// lib/Pangolin_IOWrapper/Keyframe.h:66-158), computed on the device.
#include <algorithm>
#include <cstring>

#include "capi_common.h"

using namespace lsdg;

extern "C" void lsdg_vbo_params_default(lsdg_vbo_params* p) {
  if (!p) return;
  p->scaled_th = 1e-3f;
  p->abs_th = 1e-1f;
  p->scale = 1.0f;
  p->min_near_support = 9;
}

// Scratch for n pixels: records | the filter's masks and counts | vertices.
struct ExportScratch {
  lsdg_point_dense* rec;
  void* vbo;
  lsdg_vertex* vtx;
};

static lsdg_status export_scratch(lsdg_ctx c, int w, int h, ExportScratch* out) {
  const size_t n = (size_t)w * h;
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t oRec = 0, oBlk = up(n * sizeof(lsdg_point_dense)), oVtx = oBlk + up(vbo_scratch_bytes(w, h));
  const size_t total = oVtx + up(n * sizeof(lsdg_vertex));
  if (total > c->exportCap) {
    CK(c, hipStreamSynchronize(c->stream));
    if (c->d_export) (void)hipFree(c->d_export);
    c->d_export = nullptr;
    c->exportCap = 0;
    CK(c, alloc_device(&c->d_export, total));
    c->exportCap = total;
  }
  char* b = (char*)c->d_export;
  out->rec = (lsdg_point_dense*)(b + oRec);
  out->vbo = b + oBlk;
  out->vtx = (lsdg_vertex*)(b + oVtx);
  return LSDG_OK;
}

static VboArgs vbo_args(int w, int h, float fx, float fy, float cx, float cy, const lsdg_vbo_params& p) {
  VboArgs a;
  a.w = w;
  a.h = h;
  // Keyframe.h:86-89
  a.fxi = 1 / fx;
  a.fyi = 1 / fy;
  a.cxi = -cx / fx;
  a.cyi = -cy / fy;
  a.scaledTH = p.scaled_th;
  a.absTH = p.abs_th;
  a.scale = p.scale;
  a.minNear = p.min_near_support;
  return a;
}

// Depth and image of frame f at `level` are there.
static lsdg_status exportable(lsdg_frame f, int level) {
  if (!f->hasDepth) return fail(f->ctx, LSDG_ESTATE, "keyframe has no depth");
  return frame_require(f, fd_bit(FD_IMAGE, level));
}

// Records of frame f at `level` into s.rec (device).
static lsdg_status dense_records(lsdg_frame f, int level, const ExportScratch& s) {
  lsdg_ctx c = f->ctx;
  lsdg_status st = exportable(f, level);
  if (st != LSDG_OK) return st;
  CK(c, launch_kf_dense(f->d_idepth[level], f->d_ivar[level], f->d_image[level], f->w[level] * f->h[level], s.rec,
                        c->stream));
  return LSDG_OK;
}

// The device's view of host memory that it can write (pinned), or null.
static void* device_view(void* host) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, host) != hipSuccess) {
    (void)hipGetLastError();  // ordinary host memory
    return nullptr;
  }
  return at.type == hipMemoryTypeHost ? at.devicePointer : nullptr;
}

// Runs the filter (`launch` is given where the count and the vertices go) and
// brings the kept vertices to host `out`: written there by the kernel when the
// buffer is pinned, copied after the count is known otherwise.
template <class F>
static lsdg_status run_vbo(lsdg_ctx c, const ExportScratch& s, lsdg_vertex* out, int32_t* count, F&& launch) {
  lsdg_vertex* pinned = (lsdg_vertex*)device_view(out);
  CK(c, launch((int*)c->d_result, pinned ? pinned : s.vtx));
  CK(c, hipStreamSynchronize(c->stream));
  const int total = *(const volatile int*)c->h_result;
  if (total > 0 && !pinned) {
    CK(c, hipMemcpyAsync(out, s.vtx, sizeof(lsdg_vertex) * (size_t)total, hipMemcpyDeviceToHost, c->stream));
    CK(c, hipStreamSynchronize(c->stream));
  }
  *count = total;
  return LSDG_OK;
}

extern "C" lsdg_status lsdg_keyframe_points(lsdg_frame kf, int32_t level, lsdg_point_dense* out) {
  if (!kf || !out || level < 0 || level >= PYR) return LSDG_EINVAL;
  lsdg_ctx c = kf->ctx;
  ExportScratch s;
  lsdg_status st = export_scratch(c, kf->w[level], kf->h[level], &s);
  if (st == LSDG_OK) st = dense_records(kf, level, s);
  if (st != LSDG_OK) return st;
  CK(c, hipMemcpyAsync(out, s.rec, sizeof(lsdg_point_dense) * (size_t)kf->w[level] * kf->h[level],
                       hipMemcpyDeviceToHost, c->stream));
  CK(c, hipStreamSynchronize(c->stream));
  return LSDG_OK;
}

extern "C" lsdg_status lsdg_points_vbo(lsdg_ctx c, const lsdg_point_dense* in, int32_t w, int32_t h, float fx,
                                       float fy, float cx, float cy, const lsdg_vbo_params* p, lsdg_vertex* out,
                                       int32_t* count) {
  if (!c || !in || !p || !out || !count || w < 1 || h < 1 || w > 16384 || h > 16384) return LSDG_EINVAL;
  ExportScratch s;
  lsdg_status st = export_scratch(c, w, h, &s);
  if (st != LSDG_OK) return st;
  CK(c, hipMemcpyAsync(s.rec, in, sizeof(lsdg_point_dense) * (size_t)w * h, hipMemcpyHostToDevice, c->stream));
  const VboArgs a = vbo_args(w, h, fx, fy, cx, cy, *p);
  return run_vbo(c, s, out, count,
                 [&](int* total, lsdg_vertex* v) { return launch_vbo(s.rec, a, s.vbo, total, v, c->stream); });
}

extern "C" lsdg_status lsdg_keyframe_vbo(lsdg_frame kf, int32_t level, const lsdg_vbo_params* p, lsdg_vertex* out,
                                         int32_t* count) {
  if (!kf || !p || !out || !count || level < 0 || level >= PYR) return LSDG_EINVAL;
  lsdg_ctx c = kf->ctx;
  const int w = kf->w[level], h = kf->h[level];
  ExportScratch s;
  lsdg_status st = export_scratch(c, w, h, &s);
  if (st == LSDG_OK) st = exportable(kf, level);
  if (st != LSDG_OK) return st;
  const VboArgs a = vbo_args(w, h, kf->fx[level], kf->fy[level], kf->cx[level], kf->cy[level], *p);
  return run_vbo(c, s, out, count, [&](int* total, lsdg_vertex* v) {
    return launch_vbo(kf->d_idepth[level], kf->d_ivar[level], kf->d_image[level], a, s.vbo, total, v, c->stream);
  });
}
