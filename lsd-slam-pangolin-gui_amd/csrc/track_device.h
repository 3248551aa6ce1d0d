// Per-point tracker math shared by the plain (one alignment per launch) and
// batched (many alignments per launch) evaluation kernels: bilinear taps of the
// (I, gx, gy) pyramid in FP32 / FP16 / BF16, the Jacobian row, the per-thread
// accumulators, and one function per point for SE3, Sim3 and the adjoint.
// The float expressions keep the reference's operation order (SE3Tracker::
// calcResidualAndBuffers / calcWeightsAndResidual / calculateWarpUpdate and the
// Sim3Tracker counterparts) so masks and counts match the CPU restatement.
#pragma once
#include <type_traits>

#include "lsdg_internal.h"

namespace lsdg {

constexpr int EVAL_BS = 256;
constexpr int EVAL_WAVES = EVAL_BS / 64;
constexpr int EVAL_U = 2;  // points per thread with loads in flight together (plain kernels)

struct Taps {
  float gx, gy, I;
};

__device__ inline float bf16_to_f32(unsigned short h) { return __uint_as_float(((unsigned)h) << 16); }

template <int PREC>
__device__ inline Taps load_tap(const void* img, int i) {
  if constexpr (PREC == LSDG_FP32) {
    float4 g = ((const float4*)img)[i];
    return {g.x, g.y, g.z};
  } else {
    uint2 g = ((const uint2*)img)[i];
    if constexpr (PREC == LSDG_FP16) {
      return {__half2float(__ushort_as_half((unsigned short)(g.x & 0xFFFFu))),
              __half2float(__ushort_as_half((unsigned short)(g.x >> 16))),
              __half2float(__ushort_as_half((unsigned short)(g.y & 0xFFFFu)))};
    } else {
      return {bf16_to_f32((unsigned short)(g.x & 0xFFFFu)), bf16_to_f32((unsigned short)(g.x >> 16)),
              bf16_to_f32((unsigned short)(g.y & 0xFFFFu))};
    }
  }
}

// getInterpolatedElement43: weights dxdy, dy-dxdy, dx-dxdy, 1-dx-dy+dxdy.
template <int PREC>
__device__ inline Taps interp3(const void* img, float x, float y, int w) {
  int ix = (int)x, iy = (int)y;
  float dx = x - (float)ix, dy = y - (float)iy;
  float dxdy = dx * dy;
  int b = ix + iy * w;
  Taps a11 = load_tap<PREC>(img, b + 1 + w), a01 = load_tap<PREC>(img, b + w);
  Taps a10 = load_tap<PREC>(img, b + 1), a00 = load_tap<PREC>(img, b);
  float w11 = dxdy, w01 = dy - dxdy, w10 = dx - dxdy, w00 = 1.0f - dx - dy + dxdy;
  Taps o;
  o.gx = w11 * a11.gx + w01 * a01.gx + w10 * a10.gx + w00 * a00.gx;
  o.gy = w11 * a11.gy + w01 * a01.gy + w10 * a10.gy + w00 * a00.gy;
  o.I = w11 * a11.I + w01 * a01.I + w10 * a10.I + w00 * a00.I;
  return o;
}

// Loads and stores of device memory through a pointer that the compiler only
// knows as a generic one (read from a job's descriptor): global accesses need
// no wait for the LDS queue and return in order, flat ones do neither.
template <class T>
__device__ inline T gload(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "loaded as 32-bit words");
  constexpr int N = sizeof(T) / 4;
  typedef unsigned V __attribute__((ext_vector_type(N)));
  const V v = *(const __attribute__((address_space(1))) V*)p;
  return __builtin_bit_cast(T, v);
}
__device__ inline void gstore(uint8_t* p, uint8_t v) { *(__attribute__((address_space(1))) uint8_t*)p = v; }

// The four raw taps of one bilinear sample, fetched ahead of their use so a
// thread can keep several points' loads in flight.
template <int PREC>
struct TapRaw {
  using T = typename std::conditional<PREC == LSDG_FP32, float4, uint2>::type;
  T a11, a01, a10, a00;
  float dx, dy;
};

template <int PREC>
__device__ inline Taps decode_tap(const typename TapRaw<PREC>::T& g) {
  if constexpr (PREC == LSDG_FP32) {
    return {g.x, g.y, g.z};
  } else if constexpr (PREC == LSDG_FP16) {
    return {__half2float(__ushort_as_half((unsigned short)(g.x & 0xFFFFu))),
            __half2float(__ushort_as_half((unsigned short)(g.x >> 16))),
            __half2float(__ushort_as_half((unsigned short)(g.y & 0xFFFFu)))};
  } else {
    return {bf16_to_f32((unsigned short)(g.x & 0xFFFFu)), bf16_to_f32((unsigned short)(g.x >> 16)),
            bf16_to_f32((unsigned short)(g.y & 0xFFFFu))};
  }
}

template <int PREC>
__device__ inline void fetch_taps(const void* img, float x, float y, int w, TapRaw<PREC>& t) {
  using T = typename TapRaw<PREC>::T;
  const T* im = (const T*)img;
  int ix = (int)x, iy = (int)y;
  t.dx = x - (float)ix;
  t.dy = y - (float)iy;
  const T* r0 = im + (unsigned)(ix + iy * w);
  const T* r1 = r0 + (unsigned)w;
  t.a11 = gload(r1 + 1);
  t.a01 = gload(r1);
  t.a10 = gload(r0 + 1);
  t.a00 = gload(r0);
}

// interp3's weighted sum of fetched taps (same operations, same order).
template <int PREC>
__device__ inline Taps blend_taps(const TapRaw<PREC>& t) {
  float dx = t.dx, dy = t.dy;
  float dxdy = dx * dy;
  Taps a11 = decode_tap<PREC>(t.a11), a01 = decode_tap<PREC>(t.a01);
  Taps a10 = decode_tap<PREC>(t.a10), a00 = decode_tap<PREC>(t.a00);
  float w11 = dxdy, w01 = dy - dxdy, w10 = dx - dxdy, w00 = 1.0f - dx - dy + dxdy;
  Taps o;
  o.gx = w11 * a11.gx + w01 * a01.gx + w10 * a10.gx + w00 * a00.gx;
  o.gy = w11 * a11.gy + w01 * a01.gy + w10 * a10.gy + w00 * a00.gy;
  o.I = w11 * a11.I + w01 * a01.I + w10 * a10.I + w00 * a00.I;
  return o;
}

// Division, reciprocal and square root of the per-point math.  FP32 pyramids
// use IEEE correctly rounded operations (the CPU restatement's results, bit
// for bit); FP16 / BF16 pyramids use the hardware reciprocal and square-root
// approximations (about 1 ulp, far below the taps' 11- / 8-bit quantisation),
// which cut the evaluation's VALU work by about a third.
template <int PREC>
__device__ inline float fdiv(float a, float b) {
  if constexpr (PREC == LSDG_FP32) return a / b;
  else return a * __builtin_amdgcn_rcpf(b);
}
template <int PREC>
__device__ inline float frcp(float b) {
  if constexpr (PREC == LSDG_FP32) return 1.0f / b;
  else return __builtin_amdgcn_rcpf(b);
}
template <int PREC>
__device__ inline float fsqrt(float x) {
  if constexpr (PREC == LSDG_FP32) return sqrtf(x);
  else return __builtin_amdgcn_sqrtf(x);
}

// The FP32 point math divides about ten times by six values.  A / operator is
// a scaled sequence of ten instructions each time; where the operands are far
// from the ends of the exponent range the scaling is not needed and one
// correctly rounded reciprocal serves every division by the same value.
//
// recip_rn: v_rcp_f32 is within 1 ulp; one Newton step in fma arithmetic gives
// 1 / b correctly rounded (oracle/rounding_check.hip compares all three on the
// device: reciprocals and roots of every float of the range, quotients for
// every significand of the denominator).
// div_rn: a / b from y = RN(1 / b).  q0 = RN(a y) is within two ulps; the
// remainder a - b q0 is exact up to 2^-24 of itself, so q1 is within one ulp
// of a / b, its remainder is exact, and the last fma rounds correctly
// (Markstein 1990: a faithful quotient, an exact remainder and RN(1 / b)).
// sqrt_rn: v_sqrt_f32 is within 1 ulp; s is moved to a neighbour when
// s (s - ulp) >= x or s (s + ulp) < x.
// All three need operands and results well inside the normal range, which
// exp_in / num_ok test on the wave before they are used.
// The evaluation is bound by VALU issue: about 120 of an FP32 point's 560
// instructions were the scaled sequences, of which 45 remain (64 alignments of
// 640x480 in one plan: 562 -> 534 us).
struct RecipRN {
  float b, y;
};
__device__ inline RecipRN recip_rn(float b) {
  const float y0 = __builtin_amdgcn_rcpf(b);
  return {b, __builtin_fmaf(__builtin_fmaf(-b, y0, 1.0f), y0, y0)};
}
__device__ inline float div_rn(float a, const RecipRN& r) {
  const float q0 = a * r.y;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-r.b, q0, a), r.y, q0);
  return __builtin_fmaf(__builtin_fmaf(-r.b, q1, a), r.y, q1);
}
__device__ inline float sqrt_rn(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float lo = __uint_as_float(__float_as_uint(s) - 1u), hi = __uint_as_float(__float_as_uint(s) + 1u);
  float o = __builtin_fmaf(-lo, s, x) <= 0.0f ? lo : s;
  return __builtin_fmaf(-hi, s, x) > 0.0f ? hi : o;
}
// |x| in [2^-E, 2^E]: one shift-and-add and an unsigned compare (the sign
// shifts out; zero, infinities and NaN fail).
template <int E>
__device__ inline unsigned exp_key(float x) {
  return (__float_as_uint(x) << 1) - ((127u - E) << 24);
}
template <int E>
__device__ inline bool exp_in(float x) {
  return exp_key<E>(x) <= (2u * E) << 24;
}
// x is zero or at least 2^-90 in magnitude: the remainders of its division
// stay normal numbers.
__device__ inline unsigned num_key(float x) { return (__float_as_uint(x) << 1) - (37u << 24); }
__device__ inline bool num_ok(unsigned key) { return key <= 0u - (37u << 24); }

// Projection of one reference point into the frame (the warp every tracker
// evaluation starts with).
struct Proj {
  float Wx, Wy, Wz, u, v;
  float rz;   // FP32, fast: RN(1 / Wz)
  bool fast;  // FP32: the wave's Wz and p.z allow the unscaled divisions
  bool in;
};

template <int PREC>
__device__ inline Proj project(const float4& p, const Xf& x, const LevelGeom& g) {
  const float wlim = (float)(g.w - 2), hlim = (float)(g.h - 2);
  Proj o;
  o.Wx = x.R[0] * p.x + x.R[1] * p.y + x.R[2] * p.z + x.t[0];
  o.Wy = x.R[3] * p.x + x.R[4] * p.y + x.R[5] * p.z + x.t[1];
  o.Wz = x.R[6] * p.x + x.R[7] * p.y + x.R[8] * p.z + x.t[2];
  o.fast = false;
  o.rz = 0.0f;
  if constexpr (PREC == LSDG_FP32) {
    // depths within [2^-20, 2^20] (any unit a map is kept in): every
    // denominator below stays within [2^-60, 2^60]
    o.fast = __all(max(exp_key<20>(o.Wz), exp_key<20>(p.z)) <= 40u << 24);
    if (__builtin_expect(o.fast, 1)) {
      const RecipRN r = recip_rn(o.Wz);
      o.rz = r.y;
      o.u = div_rn(o.Wx, r) * g.fx + g.cx;
      o.v = div_rn(o.Wy, r) * g.fy + g.cy;
    } else {
      o.u = (o.Wx / o.Wz) * g.fx + g.cx;
      o.v = (o.Wy / o.Wz) * g.fy + g.cy;
    }
  } else {
    o.u = fdiv<PREC>(o.Wx, o.Wz) * g.fx + g.cx;
    o.v = fdiv<PREC>(o.Wy, o.Wz) * g.fy + g.cy;
  }
  o.in = o.u > 1.0f && o.v > 1.0f && o.u < wlim && o.v < hlim;
  return o;
}

// -v = dr/dxi of the photometric residual (SE3Tracker::calculateWarpUpdate).
__device__ inline void jac6(float px, float py, float z, float z_sqr, float gx, float gy, float* v) {
  v[0] = z * gx;
  v[1] = z * gy;
  v[2] = (-px * z_sqr) * gx + (-py * z_sqr) * gy;
  v[3] = (-px * py * z_sqr) * gx + (-(1.0f + py * py * z_sqr)) * gy;
  v[4] = (1.0f + px * px * z_sqr) * gx + (px * py * z_sqr) * gy;
  v[5] = (-py * z) * gx + (px * z) * gy;
}

// The quotients every point needs of its depth before and after the warp:
// z = 1 / Wz, z_sqr = 1 / Wz^2, dc = p.z / Wz, and of the denominator
// Wz^2 / p.z the derivatives g0, g1 of the projection (and with G2 g2, of
// 1 / Wz) by the point's inverse depth.
struct PointGeom {
  float z, z_sqr, dc, g0, g1, g2;
};
template <int PREC, bool G2>
__device__ inline PointGeom point_geom(float pz, const Proj& w, const Xf& x) {
  const float n0 = x.t[0] * w.Wz - x.t[2] * w.Wx;
  const float n1 = x.t[1] * w.Wz - x.t[2] * w.Wy;
  const float n2 = G2 ? w.Wz - x.t[2] : 0.0f;
  PointGeom o;
  o.g2 = 0.0f;
  if constexpr (PREC == LSDG_FP32) {
    unsigned nk = max(num_key(n0), num_key(n1));
    if (G2) nk = max(nk, num_key(n2));
    if (__builtin_expect(w.fast && __all(num_ok(nk)), 1)) {
      o.z = w.rz;
      o.z_sqr = recip_rn(w.Wz * w.Wz).y;
      o.dc = div_rn(pz, RecipRN{w.Wz, w.rz});
      const RecipRN den = recip_rn(w.Wz * w.Wz * recip_rn(pz).y);
      o.g0 = div_rn(n0, den);
      o.g1 = div_rn(n1, den);
      if (G2) o.g2 = div_rn(n2, den);
      return o;
    }
  }
  const float d = frcp<PREC>(pz);
  o.z = frcp<PREC>(w.Wz);
  o.z_sqr = frcp<PREC>(w.Wz * w.Wz);
  o.dc = fdiv<PREC>(pz, w.Wz);
  o.g0 = fdiv<PREC>(n0, w.Wz * w.Wz * d);
  o.g1 = fdiv<PREC>(n1, w.Wz * w.Wz * d);
  if (G2) o.g2 = fdiv<PREC>(n2, w.Wz * w.Wz * d);
  return o;
}

// w = 1 / D and sqrt(w) of a variance D.
template <int PREC>
__device__ inline void weight_of(float D, float& w, float& sq) {
  if constexpr (PREC == LSDG_FP32) {
    if (__builtin_expect(__all(exp_in<60>(D)), 1)) {
      w = recip_rn(D).y;
      sq = sqrt_rn(w);
      return;
    }
  }
  w = frcp<PREC>(D);
  sq = fsqrt<PREC>(w);
}

// The Huber weight min(1, k / e) of a normalised residual e >= 0.
template <int PREC>
__device__ inline float huber_weight(float e, float k) {
  if (e < k) return 1.0f;
  if constexpr (PREC == LSDG_FP32) {
    if (__builtin_expect(__all(exp_in<60>(e) && exp_in<60>(k)), 1)) return fabsf(div_rn(k, recip_rn(e)));
  }
  return fabsf(fdiv<PREC>(k, e));
}

// a / b < 1 for a >= 0 without the division: for floats a < b the quotient is
// at most pred(b) / b <= 1 - 2^-24, a float, and rounds to no more than that;
// with b < 0 it is negative (or -0).
__device__ inline bool ratio_below_one(float a, float b) { return a < b || (b < 0.0f && a == a); }

// Per-thread accumulators of the per-point FP32 terms.
//  ACC_F64:   each FP32 term is widened and summed in FP64 (the parity mode:
//             the same terms as the CPU restatement, summed to ~1e-16).
//  ACC_KAHAN: compensated FP32.  Each thread keeps a (sum, correction) pair
//             per value and adds a term with Kahan's update (4 FP32
//             operations); the wave and block trees merge pairs with TwoSum
//             (Knuth), so a block's total is its FP32 pair widened to FP64
//             once, and only the cross-block merge runs in FP64.  The error
//             of a block total is ~2 * 2^-24 * sum |term|, independent of the
//             point count.
//  ACC_TWOSUM: the same pairs, but each term's rounding error is recovered
//             exactly (TwoSum, 7 FP32 operations) and only the corrections'
//             sum rounds: about 2^-48 * sum |term| per term of a thread.  The
//             single evaluations and alignments sum this way: their grids give
//             a thread several points, where Kahan's update, which rounds the
//             correction into the next term, loses what one point per thread
//             keeps (SE3 poses of 60 pairs up to 1280x960 came out 2e-8 on
//             average from the FP64 mode's, 6e-7 at most; now 4e-16 and 5e-15).
//             An alignment takes 4% longer for it (640x480 207 -> 215 us).
constexpr int ACC_F64 = 0;
constexpr int ACC_KAHAN = 1;
constexpr int ACC_TWOSUM = 2;

// lo + up after swapping lo's upper half-wave (offset 32) or odd rows
// (offset 16) with up's lower half-wave / even rows, 32 bits at a time
// (v_permlane32_swap / v_permlane16_swap).
__device__ inline double swap_sum(double lo, double up, int offset) {
  const unsigned long long l = (unsigned long long)__double_as_longlong(lo);
  const unsigned long long u = (unsigned long long)__double_as_longlong(up);
  unsigned l0 = (unsigned)l, l1 = (unsigned)(l >> 32), u0 = (unsigned)u, u1 = (unsigned)(u >> 32);
  if (offset == 32) {
    auto r0 = __builtin_amdgcn_permlane32_swap(l0, u0, false, false);
    auto r1 = __builtin_amdgcn_permlane32_swap(l1, u1, false, false);
    l0 = r0[0]; u0 = r0[1]; l1 = r1[0]; u1 = r1[1];
  } else {
    auto r0 = __builtin_amdgcn_permlane16_swap(l0, u0, false, false);
    auto r1 = __builtin_amdgcn_permlane16_swap(l1, u1, false, false);
    l0 = r0[0]; u0 = r0[1]; l1 = r1[0]; u1 = r1[1];
  }
  const double nl = __longlong_as_double((long long)(((unsigned long long)l1 << 32) | l0));
  const double nu = __longlong_as_double((long long)(((unsigned long long)u1 << 32) | u0));
  return nl + nu;
}

// A value from the lane that offset h of the reduce-scatters below pairs with
// this one, by data parallel primitives (no LDS round trip): h = 8 is a
// rotation of the row of 16 by 8 (lane ^ 8), 4 the mirror of half a row
// (lane ^ 7), 2 and 1 quad permutations (lane ^ 2, lane ^ 1).  lane ^ 7
// differs from the lane in bit 2, as lane ^ 4 does, which is all the halving
// needs; the pairings span the row all the same.
template <int H>
__device__ inline unsigned dpp_partner(unsigned x) {
  constexpr int CTRL = H == 8 ? 0x128 : H == 4 ? 0x141 : H == 2 ? 0x4E : 0xB1;
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false);
}
template <int H>
__device__ inline double dpp_partner(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = dpp_partner<H>((unsigned)b), hi = dpp_partner<H>((unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <int H>
__device__ inline void halve_f64(double* a, int lane) {
  const bool hi = (lane & H) != 0;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const double send = hi ? a[i] : a[i + H];
    const double keep = hi ? a[i + H] : a[i];
    a[i] = keep + dpp_partner<H>(send);
  }
}

// Reduce-scatter over the wave (NS <= 64): afterwards lane l holds the wave
// total of value l (0 for l >= NS).  Halving butterfly: at each offset a lane
// keeps one half of its values and receives the other half from its partner.
// Offsets 32 and 16 use the permlane swaps (the sum of the swapped pair is
// already the kept half: no lane selects), offsets 8..1 DPP moves.  Every
// evaluation of an alignment ends in one, on its critical path; as shuffles
// through the LDS the last four offsets waited for it four times.
template <int NS>
__device__ inline double wave_reduce_scatter_f64(const double* v) {
  static_assert(NS <= 64, "reduce-scatter holds one value per lane");
  const int lane = threadIdx.x & 63;
  double a[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) a[i] = i < NS ? swap_sum(v[i], (i + 32 < NS) ? v[i + 32] : 0.0, 32) : 0.0;
#pragma unroll
  for (int i = 0; i < 16; ++i) a[i] = swap_sum(a[i], a[i + 16], 16);
  halve_f64<8>(a, lane);
  halve_f64<4>(a, lane);
  halve_f64<2>(a, lane);
  halve_f64<1>(a, lane);
  return a[0];
}

template <int MODE, int NS>
struct Accum;

template <int NS>
struct Accum<ACC_F64, NS> {
  double v[NS];
  int n[2];  // counts, one register each until set_count
  __device__ inline void zero() {
#pragma unroll
    for (int k = 0; k < NS; ++k) v[k] = 0.0;
    n[0] = n[1] = 0;
  }
  __device__ inline void add(int k, float x) { v[k] += (double)x; }
  __device__ inline void set_count(int k, int c) { v[k] = (double)c; }
  __device__ inline double wave_slot() const { return wave_reduce_scatter_f64<NS>(v); }
  __device__ static inline double merge_waves(const double* cells, int stride, int waves) {
    double t = 0.0;
    for (int w = 0; w < waves; ++w) t += cells[(size_t)w * stride];
    return t;
  }
};

// Kahan's compensated update of the pair (s, c), whose value is s + c.
__device__ inline void kahan_add(float& s, float& c, float x) {
  const float y = x + c;
  const float t = s + y;
  c = y - (t - s);
  s = t;
}

// (s, c) += x, the sum's rounding error recovered exactly.
__device__ inline void two_sum_add(float& s, float& c, float x) {
  const float t = s + x;
  const float bp = t - s;
  c += (s - (t - bp)) + (x - bp);
  s = t;
}

// (s, c) += (s2, c2): the sums' rounding error is recovered exactly with
// TwoSum and folded into the correction.
__device__ inline void pair_merge(float& s, float& c, float s2, float c2) {
  const float t = s + s2;
  const float bp = t - s;
  const float e = (s - (t - bp)) + (s2 - bp);
  c = (c + c2) + e;
  s = t;
}

// A pair packed into one 64-bit LDS cell (low word sum, high word correction).
__device__ inline double pack_pair(float s, float c) {
  return __longlong_as_double((long long)(((unsigned long long)__float_as_uint(c) << 32) | __float_as_uint(s)));
}
__device__ inline void unpack_pair(double cell, float& s, float& c) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(cell);
  s = __uint_as_float((unsigned)b);
  c = __uint_as_float((unsigned)(b >> 32));
}

// The reduce-scatter of wave_reduce_scatter_f64 over (sum, correction) pairs:
// afterwards lane l holds the wave's pair of value l ((0, 0) for l >= NS).
template <int H>
__device__ inline void halve_pair(float* s, float* c, int lane) {
  const bool hi = (lane & H) != 0;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const float ss = hi ? s[i] : s[i + H], sc = hi ? c[i] : c[i + H];
    float ks = hi ? s[i + H] : s[i], kc = hi ? c[i + H] : c[i];
    pair_merge(ks, kc, __uint_as_float(dpp_partner<H>(__float_as_uint(ss))),
               __uint_as_float(dpp_partner<H>(__float_as_uint(sc))));
    s[i] = ks;
    c[i] = kc;
  }
}
template <int NS>
__device__ inline void wave_reduce_scatter_pair(const float* vs, const float* vc, float& rs, float& rc) {
  static_assert(NS <= 64, "reduce-scatter holds one value per lane");
  const int lane = threadIdx.x & 63;
  float s[32], c[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    float ls = i < NS ? vs[i] : 0.f, lc = i < NS ? vc[i] : 0.f;
    float us = i + 32 < NS ? vs[i + 32] : 0.f, uc = i + 32 < NS ? vc[i + 32] : 0.f;
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(ls), __float_as_uint(us), false, false);
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(lc), __float_as_uint(uc), false, false);
    s[i] = __uint_as_float(a[0]);
    c[i] = __uint_as_float(b[0]);
    pair_merge(s[i], c[i], __uint_as_float(a[1]), __uint_as_float(b[1]));
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[i]), __float_as_uint(s[i + 16]), false, false);
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(c[i]), __float_as_uint(c[i + 16]), false, false);
    s[i] = __uint_as_float(a[0]);
    c[i] = __uint_as_float(b[0]);
    pair_merge(s[i], c[i], __uint_as_float(a[1]), __uint_as_float(b[1]));
  }
  halve_pair<8>(s, c, lane);
  halve_pair<4>(s, c, lane);
  halve_pair<2>(s, c, lane);
  halve_pair<1>(s, c, lane);
  rs = s[0];
  rc = c[0];
}

template <int NS>
struct Accum<ACC_KAHAN, NS> {
  float s[NS], c[NS];
  int n[2];
  __device__ inline void zero() {
#pragma unroll
    for (int k = 0; k < NS; ++k) s[k] = c[k] = 0.f;
    n[0] = n[1] = 0;
  }
  __device__ inline void add(int k, float x) { kahan_add(s[k], c[k], x); }
  // (a thread's count is far below 2^24, so the float holds it)
  __device__ inline void set_count(int k, int c_) { s[k] = (float)c_; c[k] = 0.f; }
  // The LDS cell lane l of each wave writes for value l.
  __device__ inline double wave_slot() const {
    float rs, rc;
    wave_reduce_scatter_pair<NS>(s, c, rs, rc);
    return pack_pair(rs, rc);
  }
  // Block total of one value from its wave cells (cells[w * stride], wave
  // order), widened to FP64.
  __device__ static inline double merge_waves(const double* cells, int stride, int waves) {
    float ts, tc;
    unpack_pair(cells[0], ts, tc);
    for (int w = 1; w < waves; ++w) {
      float ws, wc;
      unpack_pair(cells[(size_t)w * stride], ws, wc);
      pair_merge(ts, tc, ws, wc);
    }
    return (double)ts + (double)tc;
  }
};

template <int NS>
struct Accum<ACC_TWOSUM, NS> : Accum<ACC_KAHAN, NS> {
  __device__ inline void add(int k, float x) { two_sum_add(this->s[k], this->c[k], x); }
};

// Which of a point's sums the caller reads.  An LM step reads neither the
// unweighted residuals nor, unless the affine brightness is estimated, the
// affine statistics; leaving them out frees 12 of the loop's registers.
constexpr int SUMS_LM = 0;         // the LM step's, no affine statistics
constexpr int SUMS_LM_AFFINE = 1;  // the LM step's, affine statistics where kp.aff_stats asks for them
constexpr int SUMS_ALL = 2;        // every slot (affine statistics where kp.aff_stats asks for them)

// Values of LDS or memory that every lane of the wave reads alike, moved to
// scalar registers: a loop over points then holds none of them in vector
// registers.
template <class T>
__device__ inline T uniform(const T& x) {
  static_assert(sizeof(T) % 4 == 0, "moved as 32-bit words");
  constexpr int N = sizeof(T) / 4;
  union {
    T t;
    unsigned w[N];
  } u;
  u.t = x;
#pragma unroll
  for (int k = 0; k < N; ++k) u.w[k] = __builtin_amdgcn_readfirstlane(u.w[k]);
  return u.t;
}

// Index of (i, j), i <= j, in the row-major upper triangle of a 7x7 matrix.
__host__ __device__ constexpr int tri7(int i, int j) { return i * 7 - i * (i - 1) / 2 + (j - i); }

// One reference point of an SE3 evaluation: warp, bounds, taps, residual,
// isGood, affine statistics, weights, Jacobian and normal-equation terms.
// Rest of one SE3 point once its projection and taps are in hand.
template <int PREC, int SUMS, class ACC>
__device__ inline void se3_finish(const float4& p, float pvar, int pidx, const Proj& w, const TapRaw<PREC>& t,
                                  const Xf& x, const LevelGeom& g, const TrackKParams& kp,
                                  uint8_t* __restrict__ isGood, ACC& acc) {
  const float Wx = w.Wx, Wy = w.Wy;
  if (!w.in) {
    if (isGood) gstore(isGood + (unsigned)pidx, 0);
    return;
  }
  Taps ri = blend_taps<PREC>(t);
  float c1 = kp.aff_a * p.w + kp.aff_b;
  float c2 = ri.I;
  float r = c1 - c2;
  if (SUMS != SUMS_LM && kp.aff_stats) {  // affine-brightness statistics (read only when that estimation is on)
    float wgt = fabsf(r) < 5.0f ? 1.0f : fdiv<PREC>(5.0f, fabsf(r));
    acc.add(S3_SXX, c1 * c1 * wgt);
    acc.add(S3_SYY, c2 * c2 * wgt);
    acc.add(S3_SX, c1 * wgt);
    acc.add(S3_SY, c2 * wgt);
    acc.add(S3_SW, wgt);
  }
  bool good = ratio_below_one(r * r, kp.max_diff_constant + kp.max_diff_grad_mult * (ri.gx * ri.gx + ri.gy * ri.gy));
  if (isGood) gstore(isGood + (unsigned)pidx, good ? 1 : 0);
  float gx = g.fx * ri.gx, gy = g.fy * ri.gy;
  const PointGeom q = point_geom<PREC, false>(p.z, w, x);
  if (good) {
    if (SUMS == SUMS_ALL) acc.add(S3_RESUNW, r * r);
    acc.add(S3_SIGNED, r);
  }
  acc.n[0] += good ? 1 : 0;
  acc.n[1] += 1;
  acc.add(S3_USAGE, q.dc < 1.0f ? q.dc : 1.0f);
  // calcWeightsAndResidual
  float s = kp.var_weight * pvar;
  float drpdd = gx * q.g0 + gy * q.g1;
  float w_p, sq_p;
  weight_of<PREC>(kp.noise2 + s * drpdd * drpdd, w_p, sq_p);
  float wr = fabsf(r * sq_p);
  float wh = huber_weight<PREC>(wr, kp.huber);
  float W = wh * w_p;
  // calculateWarpUpdate
  float jv[6];
  jac6(Wx, Wy, q.z, q.z_sqr, gx, gy, jv);
  int k = 0;
#pragma unroll
  for (int a = 0; a < 6; ++a)
#pragma unroll
    for (int c = a; c < 6; ++c) acc.add(S3_A + (k++), jv[a] * jv[c] * W);
  float rW = r * W;
#pragma unroll
  for (int a = 0; a < 6; ++a) acc.add(S3_B + a, -(jv[a] * rW));
  acc.add(S3_ERR, r * r * W);
}

// SE3 evaluation of points i, i + stride, ... < end of one thread, U points
// at a time: the U points' loads are issued, then their projections' taps,
// then the U points are finished in index order (the per-thread summation
// order of a one-point-at-a-time loop).
template <int PREC, int U, int SUMS, class ACC>
__device__ inline void se3_points(const PointsLevel& pts, int i, int stride, int end, const void* __restrict__ img,
                                  const LevelGeom& g, const Xf& x, const TrackKParams& kp,
                                  uint8_t* __restrict__ isGood, ACC& acc) {
  for (; i < end; i += U * stride) {
    float4 p[U];
    float pv[U];
    int pi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = i + u * stride;
      if (k < end) {
        p[u] = gload(pts.posI + (unsigned)k);
        pv[u] = gload(pts.var + (unsigned)k);
        pi[u] = isGood ? gload(pts.idx + (unsigned)k) : 0;
      }
    }
    Proj w[U];
    TapRaw<PREC> t[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i + u * stride < end) {
        w[u] = project<PREC>(p[u], x, g);
        if (w[u].in) fetch_taps<PREC>(img, w[u].u, w[u].v, g.w, t[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * stride < end) se3_finish<PREC, SUMS>(p[u], pv[u], pi[u], w[u], t[u], x, g, kp, isGood, acc);
  }
  acc.set_count(S3_GOOD, acc.n[0]);
  acc.set_count(S3_BAD, acc.n[1] - acc.n[0]);
  acc.set_count(S3_WARPED, acc.n[1]);
}

// Rest of one Sim3 point (photometric + depth residual) once its
// projection, taps and the frame's depth at the rounded pixel are in hand.
template <int PREC, int SUMS, class ACC>
__device__ inline void sim3_finish(const float4& p, float pvar, float2 rg, const Proj& w, const TapRaw<PREC>& t,
                                   float fidR, float varF, const Xf& x, const LevelGeom& g, const TrackKParams& kp,
                                   ACC& acc) {
  if (!w.in) return;
  const float Wx = w.Wx, Wy = w.Wy;
  Taps ri = blend_taps<PREC>(t);
  float gx, gy;
  if (kp.use_esm) {
    float rgx = kp.roll[0] * rg.x + kp.roll[1] * rg.y;
    float rgy = kp.roll[2] * rg.x + kp.roll[3] * rg.y;
    gx = g.fx * 0.5f * (ri.gx + rgx);
    gy = g.fy * 0.5f * (ri.gy + rgy);
  } else {
    gx = g.fx * ri.gx;
    gy = g.fy * ri.gy;
  }
  float c1 = kp.aff_a * p.w + kp.aff_b;
  float c2 = ri.I;
  float rp = c1 - c2;
  if (SUMS != SUMS_LM && kp.aff_stats) {
    float wgt = fabsf(rp) < 2.0f ? 1.0f : fdiv<PREC>(2.0f, fabsf(rp));
    acc.add(SM_SXX, c1 * c1 * wgt);
    acc.add(SM_SYY, c2 * c2 * wgt);
    acc.add(SM_SX, c1 * wgt);
    acc.add(SM_SY, c2 * wgt);
    acc.add(SM_SW, wgt);
  }
  const PointGeom q = point_geom<PREC, true>(p.z, w, x);
  float rd, vard;
  if (varF > 0.0f) {
    rd = q.z - fidR;
    vard = varF;
  } else {
    rd = -1.0f;
    vard = -1.0f;
  }
  acc.add(SM_USAGE, q.dc < 1.0f ? q.dc : 1.0f);
  acc.n[1] += 1;
  // calcSim3WeightsAndResidual
  float s = kp.var_weight * pvar;
  float sv = kp.var_weight * vard;
  float drpdd = gx * q.g0 + gy * q.g1;
  float w_p, w_d, sq_p, sq_d;
  weight_of<PREC>(kp.noise2 + s * drpdd * drpdd, w_p, sq_p);
  weight_of<PREC>(sv + q.g2 * q.g2 * s, w_d, sq_d);
  float wrd = fabsf(rd * sq_d);
  float wrp = fabsf(rp * sq_p);
  float wabs = sv > 0.0f ? wrd + wrp : wrp;
  float wh = huber_weight<PREC>(wabs, kp.huber);
  if (sv > 0.0f) {
    acc.add(SM_RESD, wh * w_d * rd * rd);
    acc.n[0] += 1;
  }
  acc.add(SM_RESP, wh * w_p * rp * rp);
  float wp = wh * w_p;
  float wd = sv > 0.0f ? wh * w_d : 0.0f;
  // calcSim3LGS: LGS6 over (v, w) and LGS4 over (v3, w1, w2, sigma), merged
  // into the 7x7 upper triangle at rows / columns {2, 3, 4, 6}.
  float jv[6];
  jac6(Wx, Wy, q.z, q.z_sqr, gx, gy, jv);
  float v4[4] = {q.z_sqr, q.z_sqr * Wy, -q.z_sqr * Wx, q.z};
#pragma unroll
  for (int a = 0; a < 6; ++a)
#pragma unroll
    for (int c = a; c < 6; ++c) acc.add(SM_A + tri7(a, c), jv[a] * jv[c] * wp);
  float rpW = rp * wp;
#pragma unroll
  for (int a = 0; a < 6; ++a) acc.add(SM_B + a, -(jv[a] * rpW));
  if (wd != 0.0f) {
    const int remap[4] = {2, 3, 4, 6};
    float rdW = rd * wd;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int c = a; c < 4; ++c) acc.add(SM_A + tri7(remap[a], remap[c]), v4[a] * v4[c] * wd);
      acc.add(SM_B + remap[a], -(v4[a] * rdW));
    }
  }
}

// Sim3 evaluation of points i, i + stride, ... < end of one thread, U points
// at a time (loads first, then taps and the frame depth at the rounded
// projection, then the points in index order).
template <int PREC, int U, int SUMS, class ACC>
__device__ inline void sim3_points(const PointsLevel& pts, int i, int stride, int end, const void* __restrict__ img,
                                   const float* __restrict__ fid, const float* __restrict__ fvar, const LevelGeom& g,
                                   const Xf& x, const TrackKParams& kp, ACC& acc) {
  for (; i < end; i += U * stride) {
    float4 p[U];
    float pv[U];
    float2 rg[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = i + u * stride;
      if (k < end) {
        p[u] = gload(pts.posI + (unsigned)k);
        pv[u] = gload(pts.var + (unsigned)k);
        rg[u] = kp.use_esm ? gload(pts.grad + (unsigned)k) : make_float2(0.f, 0.f);
      }
    }
    Proj w[U];
    TapRaw<PREC> t[U];
    float fd[U], fv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i + u * stride < end) {
        w[u] = project<PREC>(p[u], x, g);
        if (w[u].in) {
          fetch_taps<PREC>(img, w[u].u, w[u].v, g.w, t[u]);
          int ir = (int)(w[u].u + 0.5f) + g.w * (int)(w[u].v + 0.5f);
          fv[u] = gload(fvar + (unsigned)ir);
          fd[u] = gload(fid + (unsigned)ir);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * stride < end) sim3_finish<PREC, SUMS>(p[u], pv[u], rg[u], w[u], t[u], fd[u], fv[u], x, g, kp, acc);
  }
  acc.set_count(SM_NTD, acc.n[0]);
  acc.set_count(SM_WARPED, acc.n[1]);
}

// One reference point of the adjoint: dE/dxi into acc[0..6), E into acc[6],
// count into acc[7], dE/d(idepth) into grad_d[i].
template <int PREC, class ACC>
__device__ inline void adjoint_point(const PointsLevel& pts, int i, const void* __restrict__ img, const LevelGeom& g,
                                     const Xf& x, const TrackKParams& kp, float* __restrict__ grad_d, ACC& acc) {
  // correctly rounded divisions at every storage precision
  const float4 p = pts.posI[i];
  const float pvar = pts.var[i];
  const Proj w = project<LSDG_FP32>(p, x, g);
  if (!w.in) {
    grad_d[i] = 0.0f;
    return;
  }
  Taps ri = interp3<PREC>(img, w.u, w.v, g.w);
  float r = p.w - ri.I;
  float gx = g.fx * ri.gx, gy = g.fy * ri.gy;
  const PointGeom q = point_geom<LSDG_FP32, false>(p.z, w, x);
  float s = kp.var_weight * pvar;
  float drpdd = gx * q.g0 + gy * q.g1;
  float w_p, sq_p;
  weight_of<LSDG_FP32>(kp.noise2 + s * drpdd * drpdd, w_p, sq_p);
  float e = fabsf(r * sq_p);
  float k = kp.huber;
  float wh = huber_weight<LSDG_FP32>(e, k);
  if (k < 0.0f) wh = -wh;  // the plain quotient k / e keeps the sign of k
  acc.add(6, e < k ? 0.5f * e * e : k * e - 0.5f * k * k);
  acc.add(7, 1.0f);
  float Wr = wh * w_p * r;
  float jv[6];
  if constexpr (PREC == LSDG_FP32) jac6(w.Wx, w.Wy, q.z, q.z_sqr, gx, gy, jv);
  else jac6(w.Wx, w.Wy, frcp<PREC>(w.Wz), frcp<PREC>(w.Wz * w.Wz), gx, gy, jv);
#pragma unroll
  for (int a = 0; a < 6; ++a) acc.add(a, -(Wr * jv[a]));
  grad_d[i] = -Wr * drpdd;
}

// One reference point of the Sim3 adjoint.  E is the Sim3 tracker's
// reweighted least-squares energy with its weights frozen at x:
//   E = 1/2 sum_i wh_i (w_p,i r_p,i^2 + w_d,i r_d,i^2),
// wh the joint Huber weight, w_p / w_d the photometric / depth variance
// weights, r_d = 1/z' - idepth_frame(nearest pixel); the frame's idepth
// sample, the weights and the in-image set are constants of E.  Its twist
// gradient is Sim3Tracker::calcSim3LGS's b (unnormalised) with the frame's own
// gradient in place of the ESM average (kp.use_esm must be 0).  The
// expressions are sim3_finish's, in the same order.
//   dE/dd_i = -wh w_p r_p drpdd + wh w_d r_d g2   (g2 = d(1/z')/dd).
template <int PREC, class ACC>
__device__ inline void adjoint_point_sim3(const PointsLevel& pts, int i, const void* __restrict__ img,
                                          const float* __restrict__ fid, const float* __restrict__ fvar,
                                          const LevelGeom& g, const Xf& x, const TrackKParams& kp,
                                          float* __restrict__ grad_d, ACC& acc) {
  const float4 p = pts.posI[i];
  const float pvar = pts.var[i];
  const Proj w = project<PREC>(p, x, g);
  if (!w.in) {
    grad_d[i] = 0.0f;
    return;
  }
  const float Wx = w.Wx, Wy = w.Wy;
  Taps ri = interp3<PREC>(img, w.u, w.v, g.w);
  const int ir = (int)(w.u + 0.5f) + g.w * (int)(w.v + 0.5f);
  const float varF = fvar[ir], fidR = fid[ir];
  float gx = g.fx * ri.gx, gy = g.fy * ri.gy;
  float rp = (kp.aff_a * p.w + kp.aff_b) - ri.I;
  const PointGeom q = point_geom<PREC, true>(p.z, w, x);
  float rd, vard;
  if (varF > 0.0f) {
    rd = q.z - fidR;
    vard = varF;
  } else {
    rd = -1.0f;
    vard = -1.0f;
  }
  float s = kp.var_weight * pvar;
  float sv = kp.var_weight * vard;
  float drpdd = gx * q.g0 + gy * q.g1;
  float w_p, w_d, sq_p, sq_d;
  weight_of<PREC>(kp.noise2 + s * drpdd * drpdd, w_p, sq_p);
  weight_of<PREC>(sv + q.g2 * q.g2 * s, w_d, sq_d);
  float wrd = fabsf(rd * sq_d);
  float wrp = fabsf(rp * sq_p);
  float wabs = sv > 0.0f ? wrd + wrp : wrp;
  float wh = huber_weight<PREC>(wabs, kp.huber);
  float wp = wh * w_p;
  float wd = sv > 0.0f ? wh * w_d : 0.0f;
  acc.add(AS_EP, wp * rp * rp);
  if (sv > 0.0f) acc.add(AS_ED, wh * w_d * rd * rd);
  acc.add(AS_COUNT, 1.0f);
  float jv[6];
  jac6(Wx, Wy, q.z, q.z_sqr, gx, gy, jv);
  float rpW = rp * wp;
#pragma unroll
  for (int a = 0; a < 6; ++a) acc.add(AS_G + a, -(jv[a] * rpW));
  float gd = -rpW * drpdd;
  if (wd != 0.0f) {
    float v4[4] = {q.z_sqr, q.z_sqr * Wy, -q.z_sqr * Wx, q.z};
    const int remap[4] = {2, 3, 4, 6};
    float rdW = rd * wd;
#pragma unroll
    for (int a = 0; a < 4; ++a) acc.add(AS_G + remap[a], -(v4[a] * rdW));
    gd = gd + rdW * q.g2;
  }
  grad_d[i] = gd;
}

}  // namespace lsdg
