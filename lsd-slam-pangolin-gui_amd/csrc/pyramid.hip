// Frame pyramids and TrackingReference point clouds on gfx950.
//
//  k_pyr_images  Frame::buildImage for all levels in one launch: a block owns a
//                32x32 level-0 tile and reduces it through levels 1-4 in LDS
//                (2x2 box, ((TL + TR) + BL) + BR, times 0.25).
//  k_pyr_grads   Frame::buildGradients + buildMaxGradients for every level in
//                one launch: one thread per pixel writes (gx, gy, I, 0), the
//                optional FP16/BF16 packed copy and the 3x3 max of |grad I|
//                (recomputed from the image; identical to the reference's
//                two-pass vertical-then-horizontal max on its linear index).
//  k_pyr_depth   Frame::buildIDepthAndIDepthVar for levels 1-4 in one launch.
//  k_ingest      undistortion of an 8-bit camera image, its conversion to
//                float and buildImage's levels 1-4, in one launch.
//  k_pc_*        TrackingReference::makePointCloud as a stream compaction
//                (count, scan, write) in row-major pixel order.
#include <algorithm>

#include "lsdg_internal.h"

namespace lsdg {

struct PyrImgArgs {
  float* img[PYR];
  int w[PYR], h[PYR];
  const uint8_t* u8;  // the 8-bit level 0 when it holds the image (read instead of the float copy), or null
};

// Levels 2-4 from a block's 16x16 level-1 tile L1 (level 1 already stored).
__device__ inline void pyr_levels_2to4(const PyrImgArgs& p, const float (*L1)[17], int bx, int by) {
  __shared__ float L2[8][9];
  __shared__ float L3[4][5];
  const int t = threadIdx.x;
  if (t < 64) {
    int lx = t & 7, ly = t >> 3;
    int x = bx * 8 + lx, y = by * 8 + ly;
    float v = 0.f;
    if (x < p.w[2] && y < p.h[2]) {
      v = (L1[2 * ly][2 * lx] + L1[2 * ly][2 * lx + 1] + L1[2 * ly + 1][2 * lx] + L1[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[2][x + y * p.w[2]] = v;
    }
    L2[ly][lx] = v;
  }
  __syncthreads();
  if (t < 16) {
    int lx = t & 3, ly = t >> 2;
    int x = bx * 4 + lx, y = by * 4 + ly;
    float v = 0.f;
    if (x < p.w[3] && y < p.h[3]) {
      v = (L2[2 * ly][2 * lx] + L2[2 * ly][2 * lx + 1] + L2[2 * ly + 1][2 * lx] + L2[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[3][x + y * p.w[3]] = v;
    }
    L3[ly][lx] = v;
  }
  __syncthreads();
  if (t < 4) {
    int lx = t & 1, ly = t >> 1;
    int x = bx * 2 + lx, y = by * 2 + ly;
    if (x < p.w[4] && y < p.h[4]) {
      float v = (L3[2 * ly][2 * lx] + L3[2 * ly][2 * lx + 1] + L3[2 * ly + 1][2 * lx] + L3[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[4][x + y * p.w[4]] = v;
    }
  }
}

// Levels 1-4 of a 32x32 level-0 tile, read from the 8-bit image u8 when it
// is set or from the float level 0.
__device__ inline void pyr_images_tile(const PyrImgArgs& p, const uint8_t* __restrict__ u8, int bx, int by) {
  __shared__ float L1[16][17];
  const int t = threadIdx.x;
  const int w0 = p.w[0];
  // level 1
  {
    int lx = t & 15, ly = t >> 4;
    int x = bx * 16 + lx, y = by * 16 + ly;
    float v = 0.f;
    if (x < p.w[1] && y < p.h[1]) {
      int s = 2 * x + 2 * y * w0;
      float a, b, c, d;
      if (u8) {
        a = (float)u8[s]; b = (float)u8[s + 1]; c = (float)u8[s + w0]; d = (float)u8[s + w0 + 1];
      } else {
        const float* I = p.img[0];
        a = I[s]; b = I[s + 1]; c = I[s + w0]; d = I[s + w0 + 1];
      }
      v = (a + b + c + d) * 0.25f;
      p.img[1][x + y * p.w[1]] = v;
    }
    L1[ly][lx] = v;
  }
  __syncthreads();
  pyr_levels_2to4(p, L1, bx, by);
}

// Levels 1-4 of a 64x64 level-0 tile (the batched rebuild: a quarter of the
// blocks of the 32x32 tiling, which leaves most threads idle at the coarse
// levels), read from the 8-bit level 0 when u8 is set, else from the float
// copy.  Same operations per pixel as pyr_images_tile.
__device__ inline void pyr_images_tile64(const PyrImgArgs& p, const uint8_t* __restrict__ u8, int bx, int by) {
  __shared__ float L1[32][33];
  __shared__ float L2[16][17];
  __shared__ float L3[8][9];
  const int t = threadIdx.x;
  const int w0 = p.w[0];
  // level 1: 32x32, four pixels per thread, every load issued first.  An
  // 8-bit level 0 of even width is read as byte pairs: s is even, so both
  // rows' pairs are 2-byte aligned (the buffer itself is 256-byte aligned).
  const bool pairs = u8 && (w0 & 1) == 0;
  float q[4][4];
  bool ok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = t + 256 * i, lx = k & 31, ly = k >> 5;
    const int x = bx * 32 + lx, y = by * 32 + ly;
    ok[i] = x < p.w[1] && y < p.h[1];
    const int s = ok[i] ? 2 * x + 2 * y * w0 : 0;
    if (pairs) {
      const unsigned a = *(const unsigned short*)(u8 + s), b = *(const unsigned short*)(u8 + s + w0);
      q[i][0] = (float)(a & 0xffu); q[i][1] = (float)(a >> 8); q[i][2] = (float)(b & 0xffu); q[i][3] = (float)(b >> 8);
    } else if (u8) {
      q[i][0] = (float)u8[s]; q[i][1] = (float)u8[s + 1]; q[i][2] = (float)u8[s + w0]; q[i][3] = (float)u8[s + w0 + 1];
    } else {
      const float* I = p.img[0];
      q[i][0] = I[s]; q[i][1] = I[s + 1]; q[i][2] = I[s + w0]; q[i][3] = I[s + w0 + 1];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = t + 256 * i, lx = k & 31, ly = k >> 5;
    float v = 0.f;
    if (ok[i]) {
      v = (q[i][0] + q[i][1] + q[i][2] + q[i][3]) * 0.25f;
      p.img[1][bx * 32 + lx + (by * 32 + ly) * p.w[1]] = v;
    }
    L1[ly][lx] = v;
  }
  __syncthreads();
  {
    const int lx = t & 15, ly = t >> 4;
    const int x = bx * 16 + lx, y = by * 16 + ly;
    float v = 0.f;
    if (x < p.w[2] && y < p.h[2]) {
      v = (L1[2 * ly][2 * lx] + L1[2 * ly][2 * lx + 1] + L1[2 * ly + 1][2 * lx] + L1[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[2][x + y * p.w[2]] = v;
    }
    L2[ly][lx] = v;
  }
  __syncthreads();
  if (t < 64) {
    const int lx = t & 7, ly = t >> 3;
    const int x = bx * 8 + lx, y = by * 8 + ly;
    float v = 0.f;
    if (x < p.w[3] && y < p.h[3]) {
      v = (L2[2 * ly][2 * lx] + L2[2 * ly][2 * lx + 1] + L2[2 * ly + 1][2 * lx] + L2[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[3][x + y * p.w[3]] = v;
    }
    L3[ly][lx] = v;
  }
  __syncthreads();
  if (t < 16) {
    const int lx = t & 3, ly = t >> 2;
    const int x = bx * 4 + lx, y = by * 4 + ly;
    if (x < p.w[4] && y < p.h[4]) {
      const float v =
          (L3[2 * ly][2 * lx] + L3[2 * ly][2 * lx + 1] + L3[2 * ly + 1][2 * lx] + L3[2 * ly + 1][2 * lx + 1]) * 0.25f;
      p.img[4][x + y * p.w[4]] = v;
    }
  }
}

__global__ __launch_bounds__(256) void k_pyr_images(PyrImgArgs p) { pyr_images_tile(p, p.u8, blockIdx.x, blockIdx.y); }

// The packed word of a pixel: itself, right, below, below right.
__device__ inline uint32_t pack_quad(unsigned t0, unsigned t1, unsigned b0, unsigned b1) {
  return t0 | (t1 << 8) | (b0 << 16) | (b1 << 24);
}

// A new 8-bit image: level 0 as floats, its packed form (what the epipolar
// search samples) and levels 1-4, in one launch over 32x32 tiles.  A thread
// owns the 2x2 pixels of one level-1 pixel (sizes are even) and reads them
// and their right and lower neighbours, six loads at once, so the tile waits
// on memory once (320x240: 6.1 us for the former byte loops without the
// packed form, 4.9 us now; packing in a launch of its own took 4.3 us at
// 640x480).  Words of the last column and row, which no sample reads, repeat
// their neighbours.
__global__ __launch_bounds__(256) void k_pyr_images_u8(PyrImgArgs p, uint32_t* __restrict__ quad) {
  __shared__ float L1[16][17];
  const int t = threadIdx.x, lx = t & 15, ly = t >> 4, bx = blockIdx.x, by = blockIdx.y;
  const int w = p.w[0], h = p.h[0];
  const int x = bx * 32 + 2 * lx, y = by * 32 + 2 * ly;
  float v = 0.f;
  if (x < w && y < h) {
    const int i = x + y * w, right = x + 2 < w ? 2 : 1, below = y + 2 < h ? 2 * w : w;
    const uint8_t* u = p.u8 + i;
    const unsigned a = *(const unsigned short*)u, b = *(const unsigned short*)(u + w),
                   c = *(const unsigned short*)(u + below);
    const unsigned a2 = u[right], b2 = u[w + right], c2 = u[below + right];
    const unsigned a0 = a & 0xffu, a1 = a >> 8, b0 = b & 0xffu, b1 = b >> 8, c0 = c & 0xffu, c1 = c >> 8;
    *(float2*)(p.img[0] + i) = make_float2((float)a0, (float)a1);
    *(float2*)(p.img[0] + i + w) = make_float2((float)b0, (float)b1);
    *(uint2*)(quad + i) = make_uint2(pack_quad(a0, a1, b0, b1), pack_quad(a1, a2, b1, b2));
    *(uint2*)(quad + i + w) = make_uint2(pack_quad(b0, b1, c0, c1), pack_quad(b1, b2, c1, c2));
    v = ((float)a0 + (float)a1 + (float)b0 + (float)b1) * 0.25f;
    p.img[1][(x >> 1) + (y >> 1) * p.w[1]] = v;
  }
  L1[ly][lx] = v;
  __syncthreads();
  pyr_levels_2to4(p, L1, bx, by);
}

// Undistorter::undistort for one output pixel: the source position m (from
// the undistortion table) is bilinearly interpolated in the 8-bit input and
// truncated back to 8 bits; m.x < 0 has no source and gives 0.  Table entries
// are checked on the host (0 <= m < size - 1), so both taps are in bounds.
__device__ inline uint8_t undistort_pixel(const uint8_t* __restrict__ src, int inW, float2 m) {
  if (m.x < 0.0f) return 0;
  const int xi = (int)m.x, yi = (int)m.y;
  const float xx = m.x - (float)xi, yy = m.y - (float)yi;
  const float xxyy = xx * yy;
  const uint8_t* b = src + xi + yi * inW;
  const float v = xxyy * (float)b[1 + inW] + (yy - xxyy) * (float)b[inW] + (xx - xxyy) * (float)b[1] +
                  (1.0f - xx - yy + xxyy) * (float)b[0];
  return (uint8_t)v;
}

// InputThread's ingest of one camera image (lib/App/InputThread.cpp:59-71):
// undistortion, the 8-bit to float conversion of Frame's constructor and
// Frame::buildImage for levels 1-4, in one launch.  A block owns a 16x16
// level-0 tile (one pixel per thread: the table entry, then the source taps,
// two waits on memory), writes level 0, the 8-bit undistorted image and its
// packed form (for which it also undistorts the 33 pixels right of and below
// the tile, in the same two waits), and reduces the tile level by level in
// shared memory: a 16x16 tile holds whole 2^4 blocks of level 0, so levels
// 1-4 follow from it alone.
__global__ __launch_bounds__(256) void k_ingest(PyrImgArgs p, const uint8_t* __restrict__ src, int inW,
                                                const float2* __restrict__ map, uint8_t* __restrict__ undist,
                                                uint32_t* __restrict__ quad) {
  static_assert(PYR == 5, "a 16x16 tile holds whole 2^(PYR-1) blocks");
  __shared__ float T[16][17];
  __shared__ uint8_t U[17][20];
  const int t = threadIdx.x, lx = t & 15, ly = t >> 4;
  const int w = p.w[0], h = p.h[0];
  const int x = blockIdx.x * 16 + lx, y = blockIdx.y * 16 + ly;
  const bool inside = x < w && y < h;
  const int i = inside ? x + y * w : 0;
  // threads 0-16 take the row below, 17-32 the column to the right
  const int ex = t < 17 ? t : 16, ey = t < 17 ? 16 : t - 17;
  const int hx = blockIdx.x * 16 + ex, hy = blockIdx.y * 16 + ey;
  const bool halo = t < 33 && hx < w && hy < h;
  const float2 m = inside ? map[i] : make_float2(-1.0f, -1.0f);
  const float2 mh = halo ? map[hx + hy * w] : make_float2(-1.0f, -1.0f);
  const uint8_t u = undistort_pixel(src, inW, m);
  if (t < 33) U[ey][ex] = undistort_pixel(src, inW, mh);
  float v = 0.0f;
  if (inside) {
    v = (float)u;
    p.img[0][i] = v;
    undist[i] = u;
  }
  T[ly][lx] = v;
  U[ly][lx] = u;
  __syncthreads();
  if (inside) quad[i] = pack_quad(u, U[ly][lx + 1], U[ly + 1][lx], U[ly + 1][lx + 1]);
#pragma unroll
  for (int l = 1, n = 8; l < PYR; ++l, n >>= 1) {
    const int tx = t % n, ty = t / n;
    float c = 0.0f;
    if (t < n * n) {
      const int cx = blockIdx.x * n + tx, cy = blockIdx.y * n + ty;
      if (cx < p.w[l] && cy < p.h[l]) {
        c = (T[2 * ty][2 * tx] + T[2 * ty][2 * tx + 1] + T[2 * ty + 1][2 * tx] + T[2 * ty + 1][2 * tx + 1]) * 0.25f;
        p.img[l][cx + cy * p.w[l]] = c;
      }
    }
    __syncthreads();  // the level's reads end before its values replace them
    if (t < n * n) T[ty][tx] = c;
    __syncthreads();
  }
}

struct PyrGradArgs {
  const float* img[PYR];
  float4* grad[PYR];
  uint2* gradh[PYR];
  float* maxg[PYR];
  int w[PYR], h[PYR];
  int blk0[PYR + 1];
  int prec;
  int ppt;  // pixels per thread: a block covers ppt x 256 consecutive pixels of one level
};

__device__ inline float absgrad_at(const float* __restrict__ I, int j, int w, int h) {
  if (j >= w && j < w * (h - 1)) {
    float gx = 0.5f * (I[j + 1] - I[j - 1]);
    float gy = 0.5f * (I[j + w] - I[j - w]);
    return sqrtf(gx * gx + gy * gy);
  }
  return 0.f;
}
__device__ inline float vmax_at(const float* __restrict__ I, int j, int w, int h) {
  if (j >= w + 1 && j < w * (h - 1) - 1) {
    float g1 = absgrad_at(I, j - w, w, h), g2 = absgrad_at(I, j, w, h);
    if (g1 < g2) g1 = g2;
    float g3 = absgrad_at(I, j + w, w, h);
    return (g1 < g3) ? g3 : g1;
  }
  return 0.f;
}

__device__ inline unsigned short f32_to_bf16(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ inline uint2 pack_grad(float4 g, int prec) {
  unsigned short a, b, c;
  if (prec == LSDG_BF16) {
    a = f32_to_bf16(g.x); b = f32_to_bf16(g.y); c = f32_to_bf16(g.z);
  } else {
    a = __half_as_ushort(__float2half_rn(g.x));
    b = __half_as_ushort(__float2half_rn(g.y));
    c = __half_as_ushort(__float2half_rn(g.z));
  }
  return make_uint2((unsigned)a | ((unsigned)b << 16), (unsigned)c);
}

// Pixels per thread of the batched gradient stage (a single frame's keeps
// one per thread, for more blocks on its smaller grid).
constexpr int GRAD_PPT_BATCH = 4;

__device__ inline void pyr_grads_block(const PyrGradArgs& p, int b) {
  int l = 0;
  while (l < PYR - 1 && b >= p.blk0[l + 1]) l++;
  const int w = p.w[l], h = p.h[l];
  const float* I = p.img[l];
  // pixel i of thread t at t + 256 i
  const int base = (b - p.blk0[l]) * 256 * p.ppt + threadIdx.x;
  for (int i = 0; i < p.ppt; ++i) {
    const int idx = base + 256 * i;
    if (idx >= w * h) break;
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
    if (idx >= w && idx < w * (h - 1)) {
      g.x = 0.5f * (I[idx + 1] - I[idx - 1]);
      g.y = 0.5f * (I[idx + w] - I[idx - w]);
      g.z = I[idx];
    }
    if (p.grad[l]) p.grad[l][idx] = g;
    if (p.gradh[l]) p.gradh[l][idx] = pack_grad(g, p.prec);
    if (!p.maxg[l]) continue;
    float m;
    if (idx >= w + 1 && idx < w * (h - 1) - 1) {
      float g1 = vmax_at(I, idx - 1, w, h), g2 = vmax_at(I, idx, w, h);
      if (g1 < g2) g1 = g2;
      float g3 = vmax_at(I, idx + 1, w, h);
      m = (g1 < g3) ? g3 : g1;
    } else {
      m = absgrad_at(I, idx, w, h);
    }
    p.maxg[l][idx] = m;
  }
}

__global__ __launch_bounds__(256) void k_pyr_grads(PyrGradArgs p) { pyr_grads_block(p, blockIdx.x); }

// Batched pyramids: every frame of a batch in one launch per stage.  Block b
// belongs to the frame f with off[f] <= b < off[f + 1].
__device__ inline int frame_of_block(const int* __restrict__ off, int nf, int b) {
  int lo = 0, hi = nf - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ __launch_bounds__(256) void k_pyr_images_batch(const PyrImgArgs* __restrict__ args,
                                                          const int* __restrict__ off, const int* __restrict__ tx,
                                                          int nf) {
  int f = frame_of_block(off, nf, blockIdx.x);
  int local = blockIdx.x - off[f];
  pyr_images_tile64(args[f], args[f].u8, local % tx[f], local / tx[f]);
}

__global__ __launch_bounds__(256) void k_pyr_grads_batch(const PyrGradArgs* __restrict__ args,
                                                         const int* __restrict__ off, int nf) {
  int f = frame_of_block(off, nf, blockIdx.x);
  pyr_grads_block(args[f], blockIdx.x - off[f]);
}

__global__ __launch_bounds__(256) void k_pyr_depth(PyrDepthArgs p) {
  __shared__ float I1[16][17], V1[16][17], I2[8][9], V2[8][9], I3[4][5], V3[4][5];
  const int t = threadIdx.x, bx = blockIdx.x, by = blockIdx.y;
  const int w0 = p.w[0];
  {
    int lx = t & 15, ly = t >> 4, x = bx * 16 + lx, y = by * 16 + ly;
    float oi = -1.f, ov = -1.f;
    if (x < p.w[1] && y < p.h[1]) {
      int s = 2 * x + 2 * y * w0;
      float ia[4] = {p.id[0][s], p.id[0][s + 1], p.id[0][s + w0], p.id[0][s + w0 + 1]};
      float va[4] = {p.var[0][s], p.var[0][s + 1], p.var[0][s + w0], p.var[0][s + w0 + 1]};
      fuse4(ia, va, oi, ov);
      p.id[1][x + y * p.w[1]] = oi;
      p.var[1][x + y * p.w[1]] = ov;
    }
    I1[ly][lx] = oi;
    V1[ly][lx] = ov;
  }
  __syncthreads();
  if (t < 64) {
    int lx = t & 7, ly = t >> 3, x = bx * 8 + lx, y = by * 8 + ly;
    float oi = -1.f, ov = -1.f;
    if (x < p.w[2] && y < p.h[2]) {
      float ia[4] = {I1[2 * ly][2 * lx], I1[2 * ly][2 * lx + 1], I1[2 * ly + 1][2 * lx], I1[2 * ly + 1][2 * lx + 1]};
      float va[4] = {V1[2 * ly][2 * lx], V1[2 * ly][2 * lx + 1], V1[2 * ly + 1][2 * lx], V1[2 * ly + 1][2 * lx + 1]};
      fuse4(ia, va, oi, ov);
      p.id[2][x + y * p.w[2]] = oi;
      p.var[2][x + y * p.w[2]] = ov;
    }
    I2[ly][lx] = oi;
    V2[ly][lx] = ov;
  }
  __syncthreads();
  if (t < 16) {
    int lx = t & 3, ly = t >> 2, x = bx * 4 + lx, y = by * 4 + ly;
    float oi = -1.f, ov = -1.f;
    if (x < p.w[3] && y < p.h[3]) {
      float ia[4] = {I2[2 * ly][2 * lx], I2[2 * ly][2 * lx + 1], I2[2 * ly + 1][2 * lx], I2[2 * ly + 1][2 * lx + 1]};
      float va[4] = {V2[2 * ly][2 * lx], V2[2 * ly][2 * lx + 1], V2[2 * ly + 1][2 * lx], V2[2 * ly + 1][2 * lx + 1]};
      fuse4(ia, va, oi, ov);
      p.id[3][x + y * p.w[3]] = oi;
      p.var[3][x + y * p.w[3]] = ov;
    }
    I3[ly][lx] = oi;
    V3[ly][lx] = ov;
  }
  __syncthreads();
  if (t < 4) {
    int lx = t & 1, ly = t >> 1, x = bx * 2 + lx, y = by * 2 + ly;
    if (x < p.w[4] && y < p.h[4]) {
      float ia[4] = {I3[2 * ly][2 * lx], I3[2 * ly][2 * lx + 1], I3[2 * ly + 1][2 * lx], I3[2 * ly + 1][2 * lx + 1]};
      float va[4] = {V3[2 * ly][2 * lx], V3[2 * ly][2 * lx + 1], V3[2 * ly + 1][2 * lx], V3[2 * ly + 1][2 * lx + 1]};
      float oi, ov;
      fuse4(ia, va, oi, ov);
      p.id[4][x + y * p.w[4]] = oi;
      p.var[4][x + y * p.w[4]] = ov;
    }
  }
}

// Pixels without a usable depth become (-1, -1).
__global__ void k_depth_normalize(float* __restrict__ id, float* __restrict__ var, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float a = id[i], v = var[i];
  bool ok = isfinite(a) && v > 0.f && a > 0.f;
  if (!ok) {
    id[i] = -1.f;
    var[i] = -1.f;
  }
}

// ---------------------------------------------------------- point cloud
__device__ inline bool pc_valid(const float* id, const float* var, int idx, int w, int h) {
  int y = idx / w, x = idx - y * w;
  if (x < 1 || x >= w - 1 || y < 1 || y >= h - 1) return false;
  return !(var[idx] <= 0.f || id[idx] == 0.f);
}

// The point clouds of several levels in two launches.  A tile is PC_TILE
// consecutive pixels of one level, PC_PX per thread (pixel i of thread t at
// t + 256 i, so loads coalesce).  k_pc_count counts each tile's points;
// k_pc_write adds up the counts of the level's earlier tiles (300 integers at
// most for 640x480, read by the whole block), or on a level of more tiles
// finds them added up (TILE_SCAN_MIN), and writes its points behind them in
// row-major order.  Nothing returns to the host: the counts of points stay
// on the device beside the points, and an alignment reads them there.  (One
// count, scan and write launch and one wait for the count per level took 45 us
// a level; both launches for levels 1-4 of 640x480 take 13 us.)
constexpr int PC_PX = 4;
constexpr int PC_TILE = 256 * PC_PX;

struct PcLevel {
  const float* id;
  const float* var;
  const float* img;
  int w, h;
  float fxi, fyi, cxi, cyi;
  float4* posI;
  float* pvar;
  float2* pgrad;
  int* pidx;
  int* tiles;  // points of each tile
  int* total;  // points of the level
  int ntiles;
  int scanned;  // tiles holds the points before each tile
};
struct PcArgs {
  PcLevel lv[PYR];
  int blk0[PYR + 1];  // first block of each entry; unused entries are empty
};

__device__ inline int pc_level_of(const PcArgs& a, int b) {
  int k = 0;
  while (k < PYR - 1 && b >= a.blk0[k + 1]) ++k;
  return k;
}

__global__ __launch_bounds__(256) void k_pc_count(PcArgs a) {
  __shared__ int wc[4];
  const int k = pc_level_of(a, blockIdx.x), tile = blockIdx.x - a.blk0[k];
  const PcLevel& L = a.lv[k];
  const int n = L.w * L.h;
  int c = 0;
#pragma unroll
  for (int i = 0; i < PC_PX; ++i) {
    const int idx = tile * PC_TILE + i * 256 + (int)threadIdx.x;
    c += __popcll(__ballot(idx < n && pc_valid(L.id, L.var, idx, L.w, L.h)));
  }
  if (__lane_id() == 0) wc[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) L.tiles[tile] = wc[0] + wc[1] + wc[2] + wc[3];
}

__global__ __launch_bounds__(256) void k_pc_write(PcArgs a) {
  __shared__ int wc[PC_PX][4], before[4];
  const int k = pc_level_of(a, blockIdx.x), tile = blockIdx.x - a.blk0[k];
  const PcLevel& L = a.lv[k];
  const int n = L.w * L.h, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int part = 0;
  if (L.scanned) {
    if (threadIdx.x == 0) part = L.tiles[tile];
  } else {
    for (int t = threadIdx.x; t < tile; t += 256) part += L.tiles[t];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
  bool v[PC_PX];
  int rank[PC_PX];
#pragma unroll
  for (int i = 0; i < PC_PX; ++i) {
    const int idx = tile * PC_TILE + i * 256 + (int)threadIdx.x;
    v[i] = idx < n && pc_valid(L.id, L.var, idx, L.w, L.h);
    const unsigned long long m = __ballot(v[i]);
    rank[i] = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wc[i][wv] = __popcll(m);
  }
  if (lane == 0) before[wv] = part;
  __syncthreads();
  int base = before[0] + before[1] + before[2] + before[3];
#pragma unroll
  for (int i = 0; i < PC_PX; ++i) {
    int o = base + rank[i];
    for (int w = 0; w < 4; ++w) {
      if (w < wv) o += wc[i][w];
      base += wc[i][w];
    }
    if (!v[i]) continue;
    const int idx = tile * PC_TILE + i * 256 + (int)threadIdx.x;
    const int y = idx / L.w, x = idx - y * L.w;
    const float inv = 1.0f / L.id[idx];
    const float px = inv * (L.fxi * (float)x + L.cxi);
    const float py = inv * (L.fyi * (float)y + L.cyi);
    const float pz = inv * 1.0f;
    L.posI[o] = make_float4(px, py, pz, L.img[idx]);
    L.pvar[o] = L.var[idx];
    // the gradient k_pyr_grads stores there (points are interior pixels)
    L.pgrad[o] = make_float2(0.5f * (L.img[idx + 1] - L.img[idx - 1]), 0.5f * (L.img[idx + L.w] - L.img[idx - L.w]));
    L.pidx[o] = idx;
  }
  if (tile == L.ntiles - 1 && threadIdx.x == 0) *L.total = base;
}

// Exclusive scan of tiles[0, n) in place, their sum to *total; one block, four
// counts per thread and round.
__global__ __launch_bounds__(1024) void k_tile_scan(int* __restrict__ tiles, int n, int* __restrict__ total) {
  __shared__ int wsum[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int carry = 0;
  for (int base = 0; base < n; base += 4096) {
    const int i = base + 4 * (int)threadIdx.x;
    int v[4], own = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = i + k < n ? tiles[i + k] : 0;
      own += v[k];
    }
    int upTo = own;  // of the wave, this lane's included
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(upTo, o);
      if (lane >= o) upTo += t;
    }
    if (lane == 63) wsum[wave] = upTo;
    __syncthreads();
    int before = carry + upTo - own;
    for (int k = 0; k < 16; ++k) {
      if (k < wave) before += wsum[k];
      carry += wsum[k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i + k < n) {
        tiles[i + k] = before;
        before += v[k];
      }
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}

// ------------------------------------------------------------ launchers
hipError_t launch_tile_scan(int* tiles, int n, int* total, hipStream_t s) {
  k_tile_scan<<<dim3(1), dim3(1024), 0, s>>>(tiles, n, total);
  return hipGetLastError();
}

static PyrImgArgs pyr_img_args(lsdg_frame f) {
  PyrImgArgs p;
  for (int l = 0; l < PYR; ++l) {
    p.img[l] = f->d_image[l];
    p.w[l] = f->w[l];
    p.h[l] = f->h[l];
  }
  p.u8 = f->u8Level0 ? f->d_input_u8 : nullptr;
  return p;
}

hipError_t launch_pyr_images(lsdg_frame f, hipStream_t s) {
  const dim3 grid((f->w[0] + 31) / 32, (f->h[0] + 31) / 32);
  k_pyr_images<<<grid, dim3(256), 0, s>>>(pyr_img_args(f));
  return hipGetLastError();
}

hipError_t launch_pyr_images_u8(lsdg_frame f, hipStream_t s) {
  PyrImgArgs p = pyr_img_args(f);
  p.u8 = f->d_input_u8;
  const dim3 grid((f->w[0] + 31) / 32, (f->h[0] + 31) / 32);
  k_pyr_images_u8<<<grid, dim3(256), 0, s>>>(p, f->d_quad);
  return hipGetLastError();
}

hipError_t launch_ingest(lsdg_frame f, const uint8_t* d_src, int inW, const float2* d_map, uint8_t* d_undist,
                         hipStream_t s) {
  const dim3 grid((f->w[0] + 15) / 16, (f->h[0] + 15) / 16);
  k_ingest<<<grid, dim3(256), 0, s>>>(pyr_img_args(f), d_src, inW, d_map, d_undist, f->d_quad);
  return hipGetLastError();
}

// Fills the gradient-stage arguments of frame f for the data in `need`, ppt
// pixels per thread; returns the number of blocks (levels with nothing to
// build get none).
static int pyr_grad_args(lsdg_frame f, unsigned need, int ppt, PyrGradArgs& p) {
  p.ppt = ppt;
  int blk = 0;
  for (int l = 0; l < PYR; ++l) {
    p.img[l] = f->d_image[l];
    p.grad[l] = (need & fd_bit(FD_GRAD, l)) ? f->d_grad[l] : nullptr;
    p.gradh[l] = (need & fd_bit(FD_GRADH, l)) ? f->d_gradh[l] : nullptr;
    p.maxg[l] = (need & fd_bit(FD_MAXG, l)) ? f->d_maxg[l] : nullptr;
    p.w[l] = f->w[l];
    p.h[l] = f->h[l];
    p.blk0[l] = blk;
    if (p.grad[l] || p.gradh[l] || p.maxg[l]) blk += (f->w[l] * f->h[l] + 256 * ppt - 1) / (256 * ppt);
  }
  p.blk0[PYR] = blk;
  p.prec = f->precision;
  return blk;
}

hipError_t launch_pyr_grads(lsdg_frame f, unsigned need, hipStream_t s) {
  PyrGradArgs p;
  int blk = pyr_grad_args(f, need, 1, p);
  if (blk == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pyr_grads, dim3(blk), dim3(256), 0, s, p);
  return hipGetLastError();
}

// Host tables for the batched launches (filled once per batch plan).
size_t pyr_batch_bytes(int nf) {
  return (sizeof(PyrImgArgs) + sizeof(PyrGradArgs)) * (size_t)nf + sizeof(int) * (size_t)(3 * nf + 2) + 64;
}

// Writes the argument tables for frames fs[0..nf) into host memory `h` (laid
// out as the device copy at `d`), returns the block totals of both stages.
void pyr_batch_tables(lsdg_frame const* fs, const unsigned* need, int nf, void* h, void* d, PyrBatch* out) {
  char* hb = (char*)h;
  PyrImgArgs* ia = (PyrImgArgs*)hb;
  PyrGradArgs* ga = (PyrGradArgs*)(hb + sizeof(PyrImgArgs) * nf);
  int* ioff = (int*)(hb + (sizeof(PyrImgArgs) + sizeof(PyrGradArgs)) * nf);
  int* itx = ioff + nf + 1;
  int* goff = itx + nf;
  int ib = 0, gb = 0;
  for (int k = 0; k < nf; ++k) {
    lsdg_frame f = fs[k];
    const PyrImgArgs p = pyr_img_args(f);
    PyrGradArgs q;
    int blk = pyr_grad_args(f, need[k], GRAD_PPT_BATCH, q);
    ia[k] = p;
    ga[k] = q;
    int tx = (f->w[0] + 63) / 64, ty = (f->h[0] + 63) / 64;  // 64x64 tiles (pyr_images_tile64)
    ioff[k] = ib;
    itx[k] = tx;
    ib += tx * ty;
    goff[k] = gb;
    gb += blk;
  }
  ioff[nf] = ib;
  goff[nf] = gb;
  char* db = (char*)d;
  out->img_args = db;
  out->grad_args = db + sizeof(PyrImgArgs) * nf;
  out->img_off = (const int*)(db + (sizeof(PyrImgArgs) + sizeof(PyrGradArgs)) * nf);
  out->img_tx = out->img_off + nf + 1;
  out->grad_off = out->img_tx + nf;
  out->img_blocks = ib;
  out->grad_blocks = gb;
  out->nf = nf;
}

hipError_t launch_pyr_batch(const PyrBatch& b, hipStream_t s) {
  if (b.nf == 0) return hipSuccess;
  k_pyr_images_batch<<<dim3(b.img_blocks), dim3(256), 0, s>>>((const PyrImgArgs*)b.img_args, b.img_off, b.img_tx,
                                                               b.nf);
  if (b.grad_blocks > 0)
    k_pyr_grads_batch<<<dim3(b.grad_blocks), dim3(256), 0, s>>>((const PyrGradArgs*)b.grad_args, b.grad_off, b.nf);
  return hipGetLastError();
}

hipError_t launch_pyr_depth(lsdg_frame f, hipStream_t s) {
  PyrDepthArgs p;
  for (int l = 0; l < PYR; ++l) {
    p.id[l] = f->d_idepth[l];
    p.var[l] = f->d_ivar[l];
    p.w[l] = f->w[l];
    p.h[l] = f->h[l];
  }
  dim3 grid((f->w[0] + 31) / 32, (f->h[0] + 31) / 32);
  hipLaunchKernelGGL(k_pyr_depth, grid, dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_depth_normalize(float* id, float* var, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_depth_normalize, dim3((n + 255) / 256), dim3(256), 0, s, id, var, n);
  return hipGetLastError();
}

// Levels whose interior has more pixels than this get exactly sized point
// storage (after a wait for the count) instead of room for every pixel.
constexpr size_t PC_ROOM_MAX = (size_t)1 << 22;
static_assert(PC_ROOM_MAX >= (size_t)TILE_SCAN_MIN * PC_TILE, "levels above PC_ROOM_MAX are scanned");

static hipError_t pc_storage(lsdg_ref r, int l, size_t points) {
  if (points <= (size_t)r->cap[l] && r->d_pool[l]) return hipSuccess;
  r->ctx->blocks.put(r->d_pool[l]);  // its last readers are queued on the context's stream, as its next users will be
  r->d_pool[l] = nullptr;
  r->cap[l] = 0;
  hipError_t e = r->ctx->blocks.get(&r->d_pool[l], points * (sizeof(float4) + sizeof(float) + sizeof(float2) + sizeof(int)) + 256);
  if (e == hipSuccess) r->cap[l] = (int)points;
  return e;
}

hipError_t launch_point_clouds(lsdg_ref r, unsigned levels, hipStream_t s) {
  lsdg_frame f = r->kf;
  hipError_t e;
  int tile0[PYR + 1] = {0};
  for (int l = 0; l < PYR; ++l) tile0[l + 1] = tile0[l] + (f->w[l] * f->h[l] + PC_TILE - 1) / PC_TILE;
  if (!r->d_counts) {
    e = r->ctx->blocks.get(&r->d_counts, sizeof(int) * (PYR + tile0[PYR]));
    if (e != hipSuccess) return e;
  }
  PcArgs a;
  int nl = 0, blocks = 0, lvl[PYR];
  bool exact = false;
  for (int l = 0; l < PYR; ++l) {
    if (!(levels >> l & 1u)) continue;
    PcLevel& L = a.lv[nl];
    L.id = f->d_idepth[l];
    L.var = f->d_ivar[l];
    L.img = f->d_image[l];
    L.w = f->w[l];
    L.h = f->h[l];
    L.fxi = f->fxi[l];
    L.fyi = f->fyi[l];
    L.cxi = f->cxi[l];
    L.cyi = f->cyi[l];
    L.tiles = r->d_counts + PYR + tile0[l];
    L.total = r->d_counts + l;
    L.ntiles = tile0[l + 1] - tile0[l];
    L.scanned = L.ntiles > TILE_SCAN_MIN ? 1 : 0;
    const size_t room = (size_t)(f->w[l] - 2) * (f->h[l] - 2);
    if (room <= PC_ROOM_MAX) {
      if ((e = pc_storage(r, l, room)) != hipSuccess) return e;
    } else {
      exact = true;
    }
    a.blk0[nl] = blocks;
    blocks += L.ntiles;
    lvl[nl++] = l;
  }
  for (int k = nl; k <= PYR; ++k) a.blk0[k] = blocks;
  if (nl == 0) return hipSuccess;
  k_pc_count<<<dim3(blocks), dim3(256), 0, s>>>(a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  for (int k = 0; k < nl; ++k)
    if (a.lv[k].scanned && (e = launch_tile_scan(a.lv[k].tiles, a.lv[k].ntiles, a.lv[k].total, s)) != hipSuccess) return e;
  if (exact) {
    // a level without room for every pixel has more than TILE_SCAN_MIN tiles:
    // its count of points is there now
    int n[PYR];
    e = hipMemcpyAsync(n, r->d_counts, sizeof n, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    for (int k = 0; k < nl && e == hipSuccess; ++k) {
      const int l = lvl[k];
      if ((size_t)(f->w[l] - 2) * (f->h[l] - 2) > PC_ROOM_MAX) e = pc_storage(r, l, (size_t)std::max(n[l], 1));
    }
    if (e != hipSuccess) return e;
  }
  for (int k = 0; k < nl; ++k) {
    const int l = lvl[k];
    char* base = (char*)r->d_pool[l];
    const size_t cap = (size_t)r->cap[l];
    PointsLevel& pl = r->lv[l];
    pl.posI = (const float4*)base;
    pl.grad = (const float2*)(base + cap * sizeof(float4));
    pl.var = (const float*)(base + cap * (sizeof(float4) + sizeof(float2)));
    pl.idx = (const int*)(base + cap * (sizeof(float4) + sizeof(float2) + sizeof(float)));
    pl.n = 0;
    a.lv[k].posI = (float4*)pl.posI;
    a.lv[k].pvar = (float*)pl.var;
    a.lv[k].pgrad = (float2*)pl.grad;
    a.lv[k].pidx = (int*)pl.idx;
  }
  k_pc_write<<<dim3(blocks), dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace lsdg
