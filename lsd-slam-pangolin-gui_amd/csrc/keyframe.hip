// Keyframe export for display: the pointcloud records the reference's
// Pangolin output wrapper builds from a keyframe and the filter its viewer
// runs before uploading a vertex buffer.
//
//   k_kf_dense     PangolinOutputIOWrapper::publishKeyframe
//                  (lib/Pangolin_IOWrapper/PangolinOutputIOWrapper.cpp:81-89):
//                  idepth, idepth variance and the image as four color bytes.
//   k_vbo_count,   Keyframe::computeVbo (lib/Pangolin_IOWrapper/Keyframe.h:
//   k_vbo_write    91-142) as a stream compaction that keeps the viewer's
//                  raster order: a mask of kept pixels and their count per
//                  tile, then each tile adds up the counts before it and
//                  writes its kept pixels.  Every float expression keeps the
//                  reference's operation order (no contraction), so the
//                  vertices match a sequential loop bit for bit.
#include "lsdg_internal.h"

namespace lsdg {

// The reference's float-to-byte conversion truncates; values it leaves
// undefined (negative, >= 256, NaN) are clamped.
__device__ inline uint8_t color_byte(float v) {
  if (!(v > 0.0f)) return 0;
  if (v >= 255.0f) return 255;
  return (uint8_t)(int)v;
}

__global__ __launch_bounds__(256) void k_kf_dense(const float* __restrict__ id, const float* __restrict__ var,
                                                  const float* __restrict__ img, int n,
                                                  lsdg_point_dense* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  lsdg_point_dense p;
  p.idepth = id[i];
  p.idepth_var = var[i];
  const uint8_t c = color_byte(img[i]);
  p.color[0] = p.color[1] = p.color[2] = p.color[3] = c;
  out[i] = p;
}

// Where the filter's input comes from: the point records, or the arrays of the
// keyframe that k_kf_dense would make them from.
struct VboRecords {
  const lsdg_point_dense* in;
  __device__ float idepth(int i) const { return in[i].idepth; }
  __device__ float var(int i) const { return in[i].idepth_var; }
  __device__ void color(int i, uint8_t* c) const {
    for (int k = 0; k < 3; ++k) c[k] = in[i].color[k];
  }
};
struct VboFrame {
  const float *id, *iv, *img;
  __device__ float idepth(int i) const { return id[i]; }
  __device__ float var(int i) const { return iv[i]; }
  __device__ void color(int i, uint8_t* c) const { c[0] = c[1] = c[2] = color_byte(img[i]); }
};

template <class SRC>
__device__ inline bool vbo_keep(const SRC& in, int x, int y, const VboArgs& a) {
  const int w = a.w;
  if (x < 1 || x >= w - 1 || y < 1 || y >= a.h - 1) return false;
  const float idepth = in.idepth(x + y * w);
  if (idepth <= 0) return false;
  const float var = in.var(x + y * w);
  const float depth = 1 / idepth;
  float depth4 = depth * depth;
  depth4 *= depth4;
  if (var * depth4 > a.scaledTH) return false;
  if (var * depth4 * a.scale * a.scale > a.absTH) return false;
  if (a.minNear > 1) {
    int near = 0;
    for (int dx = -1; dx < 2; dx++)
      for (int dy = -1; dy < 2; dy++) {
        const float nid = in.idepth(x + dx + (y + dy) * w);
        if (nid > 0) {
          const float diff = nid - 1.0f / depth;
          if (diff * diff < 2 * var) near++;
        }
      }
    if (near < a.minNear) return false;
  }
  return true;
}

// A tile is VBO_TILE pixels in raster order, VBO_PX rounds of a block.
// mask[16 tile + 4 i + v] holds the kept pixels of wave v in round i.
constexpr int VBO_PX = 4;
constexpr int VBO_TILE = 256 * VBO_PX;

template <class SRC>
__global__ __launch_bounds__(256) void k_vbo_count(SRC in, VboArgs a, unsigned long long* __restrict__ mask,
                                                   int* __restrict__ tiles) {
  __shared__ int wc[4];
  const int wave = threadIdx.x >> 6;
  int c = 0;
#pragma unroll
  for (int r = 0; r < VBO_PX; ++r) {
    const int i = blockIdx.x * VBO_TILE + r * 256 + (int)threadIdx.x;
    const unsigned long long m = __ballot(i < a.w * a.h && vbo_keep(in, i % a.w, i / a.w, a));
    if (__lane_id() == 0) mask[(size_t)blockIdx.x * 16 + r * 4 + wave] = m;
    c += __popcll(m);
  }
  if (__lane_id() == 0) wc[wave] = c;
  __syncthreads();
  if (threadIdx.x == 0) tiles[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
}

// The kept pixels of a tile, behind those of the tiles before it (whose counts
// the block adds up itself, or with `scanned` finds added up).  They are
// gathered in LDS and leave in whole lines: `out` may be host memory, where a
// few vertices per store would be a bus transaction each.  A record per pixel,
// a count, a scan, a write and a copy behind a wait for the count took 51 us for
// a keyframe of 640x480; two launches and one wait take 27.
// A vertex as it is stored: 16 bytes of which only 4-byte alignment is known
// (the caller's buffer may begin anywhere in its pinned block).
typedef unsigned VertexWords __attribute__((ext_vector_type(4), aligned(4)));
template <class SRC>
__global__ __launch_bounds__(256) void k_vbo_write(SRC in, VboArgs a, const unsigned long long* __restrict__ mask,
                                                   const int* __restrict__ tiles, int scanned, int* __restrict__ total,
                                                   lsdg_vertex* __restrict__ out) {
  static_assert(sizeof(lsdg_vertex) == sizeof(uint4) && sizeof(lsdg_vertex) == sizeof(VertexWords) &&
                    alignof(lsdg_vertex) == alignof(VertexWords),
                "vertices move as 16-byte words");
  __shared__ uint4 stage[VBO_TILE];
  __shared__ int before[4];
  const int tile = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (!scanned) {
    int part = 0;
    for (int t = threadIdx.x; t < tile; t += 256) part += tiles[t];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
    if (lane == 0) before[wave] = part;
  }
  int n = 0;  // kept pixels of the tile's earlier waves and rounds, then of all
#pragma unroll
  for (int r = 0; r < VBO_PX; ++r)
    for (int v = 0; v < 4; ++v) {
      const unsigned long long m = mask[(size_t)tile * 16 + r * 4 + v];
      if (v == wave && (m >> lane & 1ull)) {
        const int i = tile * VBO_TILE + r * 256 + (int)threadIdx.x;
        const int x = i % a.w, y = i / a.w;
        const float depth = 1 / in.idepth(i);
        uint8_t c[3];
        in.color(i, c);
        lsdg_vertex o;
        o.point[0] = ((float)x * a.fxi + a.cxi) * depth;
        o.point[1] = ((float)y * a.fyi + a.cyi) * depth;
        o.point[2] = depth;
        o.color[3] = 100;
        o.color[2] = c[0];
        o.color[1] = c[1];
        o.color[0] = c[2];
        stage[n + __popcll(m & ((1ull << lane) - 1ull))] = __builtin_bit_cast(uint4, o);
      }
      n += __popcll(m);
    }
  __syncthreads();
  const int base = scanned ? tiles[tile] : before[0] + before[1] + before[2] + before[3];
  for (int k = threadIdx.x; k < n; k += 256)
    ((VertexWords*)out)[(size_t)base + k] = __builtin_bit_cast(VertexWords, stage[k]);
  if (tile == (int)gridDim.x - 1 && threadIdx.x == 0) *total = base + n;
}

// ------------------------------------------------------------ launchers
hipError_t launch_kf_dense(const float* id, const float* var, const float* img, int n, lsdg_point_dense* out,
                           hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_kf_dense<<<dim3((n + 255) / 256), dim3(256), 0, s>>>(id, var, img, n, out);
  return hipGetLastError();
}

static size_t vbo_tiles(int w, int h) { return ((size_t)w * h + VBO_TILE - 1) / VBO_TILE; }
size_t vbo_scratch_bytes(int w, int h) { return vbo_tiles(w, h) * (16 * sizeof(unsigned long long) + sizeof(int)) + 64; }

template <class SRC>
static hipError_t launch_vbo_of(const SRC& in, const VboArgs& a, void* scratch, int* total, lsdg_vertex* out,
                                hipStream_t s) {
  const size_t nt = vbo_tiles(a.w, a.h);
  unsigned long long* mask = (unsigned long long*)scratch;
  int* tiles = (int*)(mask + nt * 16);
  const int scan = nt > (size_t)TILE_SCAN_MIN ? 1 : 0;
  k_vbo_count<<<dim3((unsigned)nt), dim3(256), 0, s>>>(in, a, mask, tiles);
  if (scan) {
    hipError_t e = launch_tile_scan(tiles, (int)nt, total, s);
    if (e != hipSuccess) return e;
  }
  k_vbo_write<<<dim3((unsigned)nt), dim3(256), 0, s>>>(in, a, mask, tiles, scan, total, out);
  return hipGetLastError();
}

hipError_t launch_vbo(const lsdg_point_dense* in, const VboArgs& a, void* scratch, int* total, lsdg_vertex* out,
                      hipStream_t s) {
  return launch_vbo_of(VboRecords{in}, a, scratch, total, out, s);
}
hipError_t launch_vbo(const float* id, const float* var, const float* img, const VboArgs& a, void* scratch, int* total,
                      lsdg_vertex* out, hipStream_t s) {
  return launch_vbo_of(VboFrame{id, var, img}, a, scratch, total, out, s);
}

}  // namespace lsdg
