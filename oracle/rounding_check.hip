// The unscaled FP32 operations of the evaluation kernels (track_device.h)
// against FP64 results rounded once, which are the correctly rounded ones (53
// bits are at least 2 * 24 + 2): recip_rn and sqrt_rn over every significand
// and every exponent of the range they are used in, div_rn over every
// significand of the denominator with numerators at the edges and drawn ones.
#include "../lsd-slam-pangolin-gui_amd/csrc/track_device.h"

using namespace lsdg;

namespace {
constexpr int E = 60;                             // |exponent| of reciprocals' and roots' operands
constexpr unsigned long long SIG = 1ull << 23;    // significands
constexpr unsigned long long ALL = SIG * (2 * E + 1);
constexpr int NUMERATORS = 64;                    // per denominator

struct Tally {
  unsigned long long checked, bad;
  unsigned a, b, got, want;  // one that differs
};

__device__ float value(unsigned significand, int exponent) {
  return __uint_as_float(((unsigned)(exponent + 127) << 23) | significand);
}
__device__ unsigned mix(unsigned x) {
  x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
  return x;
}
__device__ void tally(Tally* t, unsigned long long n, unsigned long long bad) {
  atomicAdd(&t->checked, n);
  if (bad) atomicAdd(&t->bad, bad);
}
__device__ bool differs(float got, float want, float a, float b, Tally* t) {
  if (__float_as_uint(got) == __float_as_uint(want)) return false;
  t->a = __float_as_uint(a);
  t->b = __float_as_uint(b);
  t->got = __float_as_uint(got);
  t->want = __float_as_uint(want);
  return true;
}

// WHAT 0: recip_rn of both signs, 1: sqrt_rn
template <int WHAT>
__global__ __launch_bounds__(256) void k_unary(Tally* t) {
  unsigned long long n = 0, bad = 0;
  for (unsigned long long i = blockIdx.x * 256ull + threadIdx.x; i < ALL; i += gridDim.x * 256ull) {
    const float x = value((unsigned)(i & (SIG - 1)), (int)(i >> 23) - E);
    if (WHAT == 0) {
      bad += differs(recip_rn(x).y, (float)(1.0 / (double)x), x, 0.f, t);
      bad += differs(recip_rn(-x).y, (float)(1.0 / (double)-x), -x, 0.f, t);
      n += 2;
    } else {
      bad += differs(sqrt_rn(x), (float)sqrt((double)x), x, 0.f, t);
      n += 1;
    }
  }
  tally(t, n, bad);
}

__global__ __launch_bounds__(256) void k_div(Tally* t) {
  unsigned long long n = 0, bad = 0;
  for (unsigned long long i = blockIdx.x * 256ull + threadIdx.x; i < SIG; i += gridDim.x * 256ull) {
    const unsigned sb = (unsigned)i;
    for (int k = 0; k < NUMERATORS; ++k) {
      const unsigned r = mix(sb * NUMERATORS + k), s = mix(r ^ 0x9e3779b9u);
      const unsigned last = (unsigned)SIG - 1;
      // numerators' significands: the ends, the denominator's and its neighbours, drawn ones
      const unsigned sa = k == 0 ? 0u : k == 1 ? 1u : k == 2 ? last : k == 3 ? last - 1 : k == 4 ? sb
                          : k == 5 ? (sb + 1) & last : k == 6 ? (sb - 1) & last : k == 7 ? last - sb : r & last;
      const float b = value(sb, k < 16 ? 0 : (int)(s % (2 * E + 1)) - E);
      // numerators from 2^-90 on and quotients in the normal range
      const int ea = k < 16 ? 0 : (int)((s >> 8) % 151) - 90;
      const float a = (r >> 31 ? -1.0f : 1.0f) * value(sa, ea);
      const double q = (double)a / (double)b;
      if (!(fabs(q) > 0x1p-125 && fabs(q) < 0x1p127)) continue;
      ++n;
      bad += differs(div_rn(a, recip_rn(b)), (float)q, a, b, t);
    }
    const RecipRN y = recip_rn(value(sb, 0));
    ++n;
    bad += differs(div_rn(0.0f, y), 0.0f, 0.0f, y.b, t);
  }
  tally(t, n, bad);
}
}  // namespace

// what: 0 reciprocals, 1 square roots, 2 quotients.  out: how many were
// checked and differ; example: a, b, the result and the correct one of one.
extern "C" int rounding_check(int what, unsigned long long out[2], unsigned example[4]) {
  Tally* t = nullptr;
  Tally h{};
  hipError_t e = hipMalloc((void**)&t, sizeof h);
  if (e != hipSuccess) return (int)e;
  e = hipMemcpy(t, &h, sizeof h, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(t);
    return (int)e;
  }
  if (what == 0) k_unary<0><<<dim3(4096), dim3(256)>>>(t);
  else if (what == 1) k_unary<1><<<dim3(4096), dim3(256)>>>(t);
  else k_div<<<dim3(4096), dim3(256)>>>(t);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(&h, t, sizeof h, hipMemcpyDeviceToHost);
  out[0] = h.checked;
  out[1] = h.bad;
  example[0] = h.a, example[1] = h.b, example[2] = h.got, example[3] = h.want;
  (void)hipFree(t);
  return (int)e;
}
