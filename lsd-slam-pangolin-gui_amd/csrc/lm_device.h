// The Levenberg-Marquardt step of one alignment on the device, shared by the
// batched kernels and the single-alignment kernel: the reference's accept /
// reject / lambda / convergence logic (SE3Tracker::trackFrame,
// Sim3Tracker::trackFrameSim3) on one wave, every lane computing the same
// values from the job's control block in LDS.
//
// The step sits on the critical path of every iteration, on one wave, so its
// length is its count of dependent FP64 instructions.  Against the
// host form in lsdg_lie.h (used by the launch-per-evaluation tracker):
//   - the normal equations are solved unnormalised (a common factor of A and b
//     drops out), with one reciprocal per pivot;
//   - exp of a step is its power series in th^2 up to |w| = 0.5 rad, and the
//     square of half the step's beyond;
//   - products of unit quaternions are renormalised with one Newton step;
//   - the divisions by counts that only feed the result are left to the host.
//   - the values a step's decision needs are read from LDS together.
// All of it agrees with the host form to FP64 rounding.
// 64 SE3 alignments of 640x480 in one plan: 534 -> 498 us; 24 of 752x478:
// 408 -> 380 us; three stages of 16 Sim3 alignments of 640x480 (few points, so
// the step weighs most): 2105 -> 1380 us.
#pragma once
#include "batch_internal.h"

namespace lsdg {

// f^n as std::pow of floats gives it: the product in FP64, rounded once.
// (Rounded to float at every factor, a factor that is not a power of two gave
// another damping after a few rejections, and poses up to 5e-8 apart.)
__host__ __device__ inline float pow_int(float f, int n) {
  double r = 1.0;
  for (int i = 0; i < n; ++i) r *= (double)f;
  return (float)r;
}

__device__ inline int lm_lane() { return (int)(threadIdx.x & 63); }

// Orders the wave's LDS writes before its later LDS reads.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1 / d to an ulp (v_rcp_f64 and two Newton steps); 0 where |d| is not a
// normal finite number, which is how the LDL^T solve treats such a pivot.
__device__ inline double lm_rcp(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
  const double a = fabs(d);
  return a > DBL_MIN && a <= DBL_MAX ? y : 0.0;
}

// q / |q| for |q| within rounding of 1 (products and series of unit
// quaternions): one Newton step of the reciprocal square root.
__device__ inline void quat_renormalize(double* q) {
  const double n2 = __builtin_fma(q[0], q[0], __builtin_fma(q[1], q[1], __builtin_fma(q[2], q[2], q[3] * q[3])));
  if (fabs(n2 - 1.0) < 1e-7) {
    const double k = __builtin_fma(-0.5, n2, 1.5);
    for (int i = 0; i < 4; ++i) q[i] *= k;
  } else {
    quat_normalize(q);
  }
}

__device__ inline Pose lm_pose_mul(const Pose& a, const Pose& b) {
  Pose r;
  r.q[0] = a.q[3] * b.q[0] + a.q[0] * b.q[3] + a.q[1] * b.q[2] - a.q[2] * b.q[1];
  r.q[1] = a.q[3] * b.q[1] - a.q[0] * b.q[2] + a.q[1] * b.q[3] + a.q[2] * b.q[0];
  r.q[2] = a.q[3] * b.q[2] + a.q[0] * b.q[1] - a.q[1] * b.q[0] + a.q[2] * b.q[3];
  r.q[3] = a.q[3] * b.q[3] - a.q[0] * b.q[0] - a.q[1] * b.q[1] - a.q[2] * b.q[2];
  quat_renormalize(r.q);
  double M[9];
  quat_R(a.q, M);
  for (int i = 0; i < 3; ++i)
    r.t[i] = a.s * (M[3 * i] * b.t[0] + M[3 * i + 1] * b.t[1] + M[3 * i + 2] * b.t[2]) + a.t[i];
  r.s = a.s * b.s;
  return r;
}

// Coefficients of the power series in th^2 <= 1/4, to 2^-53, highest power
// first: sin(th) / th, cos(th), (1 - cos th) / th^2, (th - sin th) / th^3; then
// 1 / k for k = 1 ... 17 and 1 / k! for k = 15 ... 2.  They are read through a
// pointer that the compiler cannot follow: as literals it moves them out of
// the iteration into registers, where they cost the loop over the points its
// occupancy.
constexpr int LM_SIN = 0, LM_COS = 7, LM_B = 14, LM_C = 21, LM_RECIP = 28, LM_FACT = 45, LM_COEFS = 59;
static __constant__ double lm_coef_table[LM_COEFS] = {
    1.0 / 6227020800.0, -1.0 / 39916800.0, 1.0 / 362880.0, -1.0 / 5040.0, 1.0 / 120.0, -1.0 / 6.0, 1.0,
    1.0 / 479001600.0, -1.0 / 3628800.0, 1.0 / 40320.0, -1.0 / 720.0, 1.0 / 24.0, -0.5, 1.0,
    1.0 / 87178291200.0, -1.0 / 479001600.0, 1.0 / 3628800.0, -1.0 / 40320.0, 1.0 / 720.0, -1.0 / 24.0, 0.5,
    1.0 / 1307674368000.0, -1.0 / 6227020800.0, 1.0 / 39916800.0, -1.0 / 362880.0, 1.0 / 5040.0, -1.0 / 120.0,
    1.0 / 6.0,
    1.0, 1.0 / 2, 1.0 / 3, 1.0 / 4, 1.0 / 5, 1.0 / 6, 1.0 / 7, 1.0 / 8, 1.0 / 9, 1.0 / 10, 1.0 / 11, 1.0 / 12,
    1.0 / 13, 1.0 / 14, 1.0 / 15, 1.0 / 16, 1.0 / 17,
    1.0 / 1307674368000.0, 1.0 / 87178291200.0, 1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0,
    1.0 / 3628800.0, 1.0 / 362880.0, 1.0 / 40320.0, 1.0 / 5040.0, 1.0 / 720.0, 1.0 / 120.0, 1.0 / 24.0, 1.0 / 6.0,
    0.5};
typedef const __attribute__((address_space(4))) double* LmCoef;
__device__ inline LmCoef lm_coef() {
  LmCoef c = (LmCoef)lm_coef_table;
  asm volatile("" : "+s"(c));
  return c;
}

__device__ inline double horner7(double x, LmCoef c) {
  double r = c[0];
#pragma unroll
  for (int k = 1; k < 7; ++k) r = __builtin_fma(x, r, c[k]);
  return r;
}
constexpr double LM_SERIES_TH2 = 0.25;
__device__ inline void exp_q_series(const double* w, double th2, double* q, LmCoef c) {
  const double h = 0.25 * th2;  // (th / 2)^2
  const double k = 0.5 * horner7(h, c + LM_SIN);
  q[0] = k * w[0]; q[1] = k * w[1]; q[2] = k * w[2];
  q[3] = horner7(h, c + LM_COS);
  quat_renormalize(q);
}

// exp of twists outside the series' range: exp(xi) = exp(xi / 2^k)^(2^k).
constexpr int LM_MAX_HALVINGS = 64;

__device__ inline Pose lm_se3_exp(const double* xi) {
  const LmCoef cf = lm_coef();
  double v[3] = {xi[0], xi[1], xi[2]}, w[3] = {xi[3], xi[4], xi[5]};
  double th2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
  int halvings = 0;
  for (; th2 > LM_SERIES_TH2 && halvings < LM_MAX_HALVINGS; ++halvings, th2 *= 0.25)
    for (int k = 0; k < 3; ++k) v[k] *= 0.5, w[k] *= 0.5;
  Pose r;
  exp_q_series(w, th2, r.q, cf);
  apply_abc(1.0, horner7(th2, cf + LM_B), horner7(th2, cf + LM_C), w, v, r.t);
  r.s = 1.0;
  for (; halvings > 0; --halvings) r = lm_pose_mul(r, r);
  return r;
}

// exp of a sim3 twist.  V's coefficients are integrals of e^{u sg} u^k over
// [0, 1], I_k: A = I_0, B = sum_m (-1)^m th^2m I_{2m+1} / (2m+1)!,
// C = sum_m (-1)^m th^2m I_{2m+2} / (2m+2)!; downwards
// I_{k-1} = (e^sg - sg I_k) / k is stable and forgets its start
// (I_16 ~ e^sg / 17) by sg^16 / 16!.
__device__ inline Pose lm_sim3_exp(const double* xi) {
  const LmCoef cf = lm_coef();
  double v[3] = {xi[0], xi[1], xi[2]}, w[3] = {xi[3], xi[4], xi[5]};
  double sg = xi[6];
  double th2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
  int halvings = 0;
  for (; (th2 > LM_SERIES_TH2 || fabs(sg) > 0.5) && halvings < LM_MAX_HALVINGS; ++halvings, th2 *= 0.25, sg *= 0.5)
    for (int k = 0; k < 3; ++k) v[k] *= 0.5, w[k] *= 0.5;
  Pose r;
  exp_q_series(w, th2, r.q, cf);
  double es = cf[LM_FACT];
#pragma unroll
  for (int k = 1; k < 14; ++k) es = __builtin_fma(sg, es, cf[LM_FACT + k]);
  es = __builtin_fma(sg, __builtin_fma(sg, es, 1.0), 1.0);
  // b and c take I_1 ... I_14 one at a time, downwards
  double I = es * cf[LM_RECIP + 16], b = 0.0, c = 0.0;
#pragma unroll
  for (int k = 16; k >= 1; --k) {
    I = __builtin_fma(-sg, I, es) * cf[LM_RECIP + k - 1];  // I_{k-1}
    if (k - 1 >= 1 && k - 1 <= 14) {
      if ((k - 1) & 1) b = __builtin_fma(th2, b, I * cf[LM_SIN + 6 - (k - 2) / 2]);
      else c = __builtin_fma(th2, c, I * cf[LM_B + 6 - (k - 3) / 2]);
    }
  }
  apply_abc(I, b, c, w, v, r.t);
  r.s = es;
  for (; halvings > 0; --halvings) r = lm_pose_mul(r, r);
  return r;
}

// LDL^T solve of the symmetric N x N system whose upper triangle is A
// (row-major), diagonal scaled by f; pivots without a reciprocal give zero
// components, as in ldlt_solve.
template <int N>
__device__ inline void lm_solve(const double* __restrict__ A, const double* __restrict__ b, double f, double* x) {
  double U[N][N], L[N][N], inv[N], y[N];
  int o = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    // column j of the lower triangle = row j of the upper one
#pragma unroll
    for (int i = j; i < N; ++i) {
      double v = A[o + i - j];
      if (i == j) v *= f;
#pragma unroll
      for (int k = 0; k < j; ++k) v = __builtin_fma(-U[i][k], L[j][k], v);
      U[i][j] = v;
    }
    o += N - j;
    inv[j] = lm_rcp(U[j][j]);
#pragma unroll
    for (int i = j + 1; i < N; ++i) L[i][j] = U[i][j] * inv[j];
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double v = b[i];
#pragma unroll
    for (int k = 0; k < i; ++k) v = __builtin_fma(-L[i][k], y[k], v);
    y[i] = v;
  }
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
    double v = y[i] * inv[i];
#pragma unroll
    for (int k = i + 1; k < N; ++k) v = __builtin_fma(-L[k][i], x[k], v);
    x[i] = v;
  }
}

// ------------------------------------------------------------ LM steps
__device__ inline void set_eval_pose(JobState& s, const Pose& T, bool sim3) {
  pose_rt_f(T, sim3, s.xf.R, s.xf.t);
  if (sim3) pose_roll_f(T, s.roll);
}

// remaining may be null: blocks that repeat another block's LM step (the
// cooperative kernel) leave the count to that block.
__device__ inline void finish_job(JobState& s, int status, int* ntNext, int* remaining) {
  s.status = status;
  *ntNext = 0;
  if (remaining && lm_lane() == 0) atomicSub(remaining, 1);
}

// Solve (A diag*(1+lambda)) inc = b and propose Tn = exp(inc) T; lgs holds
// the upper triangle of A, then b (an evaluation's sums, or the control
// block's lgs).  Returns false when a Sim3 step diverges (|inc|^2 not in
// [0, 1)).
template <int KIND>
__device__ inline bool solve_and_propose(JobState& __restrict__ s, const double* __restrict__ lgs, const Pose& T,
                                         float lambda) {
  constexpr int N = KIND == LSDG_JOB_SIM3 ? 7 : 6;
  constexpr int NA = N * (N + 1) / 2;
  double A[NA], b[N], inc[N];
#pragma unroll
  for (int k = 0; k < NA; ++k) A[k] = lgs[k];
#pragma unroll
  for (int a = 0; a < N; ++a) b[a] = -lgs[NA + a];
  lm_solve<N>(A, b, 1.0 + (double)lambda, inc);
  double dd = 0;
  for (int a = 0; a < N; ++a) dd += inc[a] * inc[a];
  s.incSq = dd;
  if (KIND == LSDG_JOB_SIM3) {
    if (!(dd >= 0 && dd < 1)) return false;
    s.Tn = lm_pose_mul(lm_sim3_exp(inc), T);
  } else {
    s.Tn = lm_pose_mul(lm_se3_exp(inc), T);
  }
  s.phase = 1;
  set_eval_pose(s, s.Tn, KIND == LSDG_JOB_SIM3);
  return true;
}

// Keeps the evaluation's unnormalised LGS (the upper triangle and b) as the
// accepted pose's normal equations.
template <int KIND>
__device__ inline void store_lgs(JobState& __restrict__ s, const double* __restrict__ S) {
  constexpr int NL = KIND == LSDG_JOB_SIM3 ? 35 : 27;
  static_assert(SM_A == 0 && SM_B == 28 && S3_A == 0 && S3_B == 21, "b follows the triangle");
  const int lane = lm_lane();
  if (lane < NL) s.lgs[lane] = S[lane];
}

template <int KIND>
__device__ inline void begin_level(JobState& s, const JobDesc& jd, const LmParams& P, int lvl, int* ntNext,
                                   int* remaining) {
  if (KIND == LSDG_JOB_SIM3) {
    while (lvl >= jd.finalLevel && P.lv[lvl].maxIts == 0) lvl--;
  }
  if (lvl < jd.finalLevel) {
    if (KIND == LSDG_JOB_SIM3 && !s.upToDate) {
      // a final evaluation at the accepted pose for the information matrix
      s.level = jd.finalLevel;
      s.phase = 2;
      set_eval_pose(s, s.T, true);
      *ntNext = jd.lv[s.level].ntiles;
      return;
    }
    if (KIND == LSDG_JOB_SIM3 && s.T.s <= 0) {
      finish_job(s, 3, ntNext, remaining);
      return;
    }
    finish_job(s, 1, ntNext, remaining);
    return;
  }
  s.level = lvl;
  s.phase = 0;
  set_eval_pose(s, s.T, KIND == LSDG_JOB_SIM3);
  *ntNext = jd.lv[lvl].ntiles;
}

// One LM step of an SE3 job, after the evaluation whose sums are S.  Every
// value the decision needs is read in one go at the top (an LDS round trip
// each in the branches would be most of the step), and the accepted
// evaluation's equations are solved from S itself, not from the copy kept for
// later rejections.
__device__ inline void lm_step_se3(JobState& __restrict__ s, const JobDesc& __restrict__ jd,
                                   const double* __restrict__ S, const LmParams& __restrict__ P, int* ntNext,
                                   int* remaining) {
  const int lvl = s.level, phase = s.phase, itStart = s.iteration;
  const JobLevel& L = jd.lv[lvl];
  const double warped = S[S3_WARPED], sumErr = S[S3_ERR], lastErr = s.lastErr, incSq = s.incSq;
  float lambda = s.lambda;
  int incTry = s.incTry, iteration = itStart;
  const LmLevel Q = P.lv[lvl];
  const int affine = P.affine;
  const float lim = P.lim * (float)(L.g.w * L.g.h);
  Pose T = s.T;
  const Pose Tn = s.Tn;
  s.evals++;
  s.evalsAt[lvl]++;
  s.good = S[S3_GOOD];
  s.bad = S[S3_BAD];
  s.signedRes = S[S3_SIGNED];
  s.usageSum = S[S3_USAGE];
  s.usageN = L.pts.n;
  // the affine iterate is read only when the affine brightness is estimated
  if (affine) {
    const double sxx = S[S3_SXX], syy = S[S3_SYY], sx = S[S3_SX], sy = S[S3_SY], sw = S[S3_SW];
    s.affAIt = (float)sqrt((syy - sy * sy / sw) / (sxx - sx * sx / sw));
    s.affBIt = (float)((sy - (double)s.affAIt * sx) / sw);
  }
  if ((float)warped < lim) {
    finish_job(s, 2, ntNext, remaining);
    return;
  }
  const double err = sumErr / warped;
  s.numRes[lvl]++;
  bool next = false, keep = true;  // go to the next level; this evaluation's LGS is the accepted pose's
  if (phase == 0) {
    if (affine) { s.affA = s.affAIt; s.affB = s.affBIt; }
    s.lastErr = err;
    lambda = Q.lambdaInitial;
    iteration = 0;
    next = Q.maxIts <= 0;
  } else if (err < lastErr) {
    T = Tn;
    s.T = Tn;
    if (affine) { s.affA = s.affAIt; s.affB = s.affBIt; }
    const bool conv = err / lastErr > Q.convergenceEps;
    s.lastResidual = s.lastErr = err;
    lambda = lambda <= 0.2f ? 0.0f : lambda * Q.lambdaSuccess;
    iteration++;
    next = conv || iteration >= Q.maxIts;
  } else {
    next = !(incSq > Q.stepSizeMin);
    keep = false;
    if (!next) lambda = lambda == 0.0f ? 0.2f : lambda * pow_int(Q.lambdaFail, incTry);
  }
  s.lambda = lambda;
  s.iteration = iteration;
  if (next) {
    begin_level<LSDG_JOB_SE3>(s, jd, P, lvl - 1, ntNext, remaining);
    return;
  }
  if (keep) {
    s.numWarp[lvl]++;
    incTry = 0;
  }
  s.incTry = incTry + 1;
  solve_and_propose<LSDG_JOB_SE3>(s, keep ? S : s.lgs, T, lambda);
  if (keep) store_lgs<LSDG_JOB_SE3>(s, S);
  *ntNext = L.ntiles;
}

__device__ inline void sim3_res(const double* S, double* r) {
  // r = {sumResD, sumResP, numTermsD, numTermsP, set, 0, mean}; the two
  // part means are the host's to divide
  r[0] = S[SM_RESD];
  r[1] = S[SM_RESP];
  r[2] = S[SM_NTD];
  r[3] = S[SM_WARPED];
  r[4] = 1.0;
  r[5] = 0.0;
  r[6] = (S[SM_RESD] + S[SM_RESP]) / (S[SM_NTD] + S[SM_WARPED]);
}

// One LM step of a Sim3 job (see lm_step_se3).
__device__ inline void lm_step_sim3(JobState& __restrict__ s, const JobDesc& __restrict__ jd,
                                    const double* __restrict__ S, const LmParams& __restrict__ P, int* ntNext,
                                    int* remaining) {
  const int lvl = s.level, phase = s.phase;
  const JobLevel& L = jd.lv[lvl];
  const double warped = S[SM_WARPED], incSq = s.incSq, lastMean = s.lastRes[6];
  float lambda = s.lambda;
  int incTry = s.incTry, iteration = s.iteration;
  const LmLevel Q = P.lv[lvl];
  const float lim = 0.5f * P.lim * (float)(L.g.w * L.g.h);
  Pose T = s.T;
  const Pose Tn = s.Tn;
  s.evals++;
  s.evalsAt[lvl]++;
  s.usageSum = S[SM_USAGE];
  s.usageN = L.pts.n;
  if (phase == 2) {
    // final evaluation for lastSim3Hessian
    sim3_res(S, s.finalRes);
    store_lgs<LSDG_JOB_SIM3>(s, S);
    s.upToDate = 1;
    finish_job(s, T.s <= 0 ? 3 : 1, ntNext, remaining);
    return;
  }
  if ((float)warped < lim || warped < 10) {
    finish_job(s, 2, ntNext, remaining);
    return;
  }
  double res[7];
  sim3_res(S, res);
  s.numRes[lvl]++;
  bool next = false, keep = true;  // go to the next level; this evaluation's LGS is the accepted pose's
  if (phase == 0) {
    for (int k = 0; k < 7; ++k) s.lastRes[k] = res[k];
    lambda = Q.lambdaInitial;
    iteration = 0;
  } else if (res[6] < lastMean) {
    T = Tn;
    s.T = Tn;
    s.upToDate = 0;
    const bool conv = res[6] / lastMean > Q.convergenceEps;
    for (int k = 0; k < 7; ++k) s.finalRes[k] = s.lastRes[k] = res[k];
    lambda = lambda <= 0.2f ? 0.0f : lambda * Q.lambdaSuccess;
    iteration++;
    next = conv || iteration >= Q.maxIts;
  } else {
    next = !(incSq > Q.stepSizeMin);
    keep = false;
    if (!next) lambda = lambda == 0.0f ? 0.2f : lambda * pow_int(Q.lambdaFail, incTry);
  }
  s.lambda = lambda;
  s.iteration = iteration;
  if (next) {
    begin_level<LSDG_JOB_SIM3>(s, jd, P, lvl - 1, ntNext, remaining);
    return;
  }
  if (keep) {
    s.upToDate = 1;
    s.numWarp[lvl]++;
    incTry = 0;
  }
  s.incTry = incTry + 1;
  const bool ok = solve_and_propose<LSDG_JOB_SIM3>(s, keep ? S : s.lgs, T, lambda);
  if (keep) store_lgs<LSDG_JOB_SIM3>(s, S);
  if (!ok) {
    wave_sync();
    for (int k = 0; k < 28; ++k) s.lgs[k] = 0.0;
    finish_job(s, 2, ntNext, remaining);
    return;
  }
  *ntNext = L.ntiles;
}

// Start state of a job: T = (frameToRef_init)^-1, first level, counters zero.
__device__ inline void lm_begin(JobState& s, const JobDesc& jd, const LmParams& P, int* ntNext, int* remaining) {
  s = JobState{};
  s.T = pose_inv(jd.init);
  if (jd.kind == LSDG_JOB_SE3) s.T.s = 1.0;
  s.affA = 1.0f;
  s.affB = 0.0f;
  if (jd.kind == LSDG_JOB_SIM3) begin_level<LSDG_JOB_SIM3>(s, jd, P, jd.startLevel, ntNext, remaining);
  else begin_level<LSDG_JOB_SE3>(s, jd, P, jd.startLevel, ntNext, remaining);
}

// The points [begin, end) of part `part` of `parts`: contiguous, whole and
// within one of each other.
struct PartRange {
  int begin, end;
};
__device__ inline PartRange part_range(int n, int part, int parts) {
  const int q = n / parts, r = n - q * parts;
  const int b = part * q + min(part, r);
  return {b, b + q + (part < r ? 1 : 0)};
}

// Copies a trivially copyable object between global memory and LDS with the
// whole block (32-bit words).
template <class T>
__device__ inline void block_copy(T* dst, const T* src, int nthreads) {
  static_assert(sizeof(T) % 4 == 0, "copied as 32-bit words");
  const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
  uint32_t* d = reinterpret_cast<uint32_t*>(dst);
  for (int w = threadIdx.x; w < (int)(sizeof(T) / 4); w += nthreads) d[w] = s[w];
}

}  // namespace lsdg
