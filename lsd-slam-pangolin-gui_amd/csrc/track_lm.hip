// One alignment's whole Levenberg-Marquardt loop in one launch
// (SE3Tracker::trackFrame, Sim3Tracker::trackFrameSim3): what lsdg_se3_track
// and lsdg_sim3_track run.
//
// A launch per evaluation costs its kernel (about 11 us, of which the
// evaluation itself is a third: the rest is the start of the launch, the
// merge behind a completion counter and the result's way to the host) and
// about as much again for the launch, the wait and the host's LM step: 22 us
// for each of about 28 evaluations.  Here the blocks stay: every block
// reduces its range of the level's points to an FP64 row, publishes it as
// tagged words and reads the others' rows (k_batch_coop's exchange), and
// repeats the same LM step on its own copy of the control block, so an
// iteration is one evaluation, one exchange and one LM step.
//
// 320x240 camera image to pose: 725 -> 206 us; 640x480 through the
// undistorter: 638 -> 259 us (the launch itself about 170 us for 28
// evaluations: 1.4-2 us of points, 2-2.5 us of exchange and 1.3 us of LM step
// each).
//
// Blocks: track_lm_blocks.  On a small level every block evaluates the whole
// level itself and nothing is exchanged.  The blocks must be resident
// together.  They are when the device
// has that many free slots (it holds several hundred); other work on it can
// keep some of them out, so every wait is bounded, the blocks that waited in
// vain stop, and the caller runs the alignment launch by launch instead.
#include <cmath>

#include "lm_device.h"
#include "track_device.h"

namespace lsdg {

constexpr int TRACK_LM_BS = 256;
constexpr int TRACK_LM_WAVES = TRACK_LM_BS / 64;
// Levels of at most this many points are evaluated whole by every block: two
// points per thread cost less than an exchange (320x240: 162 us per alignment,
// with 1024 points 169).
constexpr int TRACK_LM_SOLO = 512;

template <int KIND, int PREC, int ACC>
__global__ __launch_bounds__(TRACK_LM_BS) void k_track_lm(TrackLmArgs a) {
  constexpr int NS = KIND == LSDG_JOB_SIM3 ? NS_SIM3 : NS_SE3;
  __shared__ JobState s;
  __shared__ JobDesc jd;
  __shared__ LmParams sP;
  __shared__ double sh[TRACK_LM_WAVES][NS];
  __shared__ double S[NS];
  __shared__ int failed;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, part = blockIdx.x;
  block_copy(&jd, &a.jd, TRACK_LM_BS);
  block_copy(&sP, &a.P, TRACK_LM_BS);
  if (tid == 0) failed = 0;
  __syncthreads();
  if (tid < 64) {
    // the counts of levels outside the job's are never read
    if (tid < PYR) jd.lv[tid].pts.n = a.counts[tid];
    wave_sync();
    int nt = 0;
    lm_begin(s, jd, sP, &nt, nullptr);
    wave_sync();
    if (tid < PYR) s.npts[tid] = jd.lv[tid].pts.n;
  }
  __syncthreads();
  // every block takes part in every exchange: one that only read could be
  // overtaken by the others' next rows
  const int parts = a.blocks;
  JobLevel L{};  // of level cur, as are split, i0 and i1 (in scalar registers)
  int cur = -1, i0 = 0, i1 = 0;
  bool split = false;
  unsigned gen = 0;  // exchanges so far
  for (int it = 0; it < BATCH_JOB_MAX_EVALS; ++it) {
    // s is read after a barrier: the exit test is uniform over the block
    if (s.status != 0) break;
    const int lvl = uniform(s.level);
    if (lvl != cur) {
      cur = lvl;
      L = uniform(jd.lv[lvl]);
      split = parts > 1 && L.pts.n > TRACK_LM_SOLO;
      const PartRange r = split ? part_range(L.pts.n, part, parts) : PartRange{0, L.pts.n};
      i0 = r.begin;
      i1 = r.end;
    }
    const Xf x = uniform(s.xf);
    TrackKParams kp = a.kp;
    kp.aff_a = uniform(s.affA);
    kp.aff_b = uniform(s.affB);
    Accum<ACC, NS> acc;
    acc.zero();
    if (KIND == LSDG_JOB_SIM3) {
      for (int k = 0; k < 4; ++k) kp.roll[k] = uniform(s.roll[k]);
      sim3_points<PREC, EVAL_U, SUMS_LM_AFFINE>(L.pts, i0 + tid, TRACK_LM_BS, i1, L.img, L.fid, L.fvar, L.g, x, kp, acc);
    } else {
      uint8_t* mask = lvl == 1 ? uniform(jd.isGood) : nullptr;
      se3_points<PREC, EVAL_U, SUMS_LM_AFFINE>(L.pts, i0 + tid, TRACK_LM_BS, i1, L.img, L.g, x, kp, mask, acc);
    }
    const double wsum = acc.wave_slot();
    if (lane < NS) sh[wave][lane] = wsum;
    __syncthreads();
    if (!split) {
      if (tid < NS) S[tid] = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, TRACK_LM_WAVES);
      __syncthreads();
    } else {
      unsigned long long* buf = a.rows + (size_t)(gen & 1) * a.blocks * NS * 2;
      const unsigned tag = a.epochTag | (gen & 0xFFFFu);
      if (tid < NS) {
        const double v = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, TRACK_LM_WAVES);
        const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
        unsigned long long* w = buf + ((size_t)part * NS + tid) * 2;
        const unsigned long long t64 = (unsigned long long)tag << 32;
        __hip_atomic_store(w, t64 | (bits & 0xFFFFFFFFull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 1, t64 | (bits >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();  // sh is read above and written below
      // each wave reads a quarter of the rows and adds them in part order
      const int q0 = parts * wave / TRACK_LM_WAVES, q1 = parts * (wave + 1) / TRACK_LM_WAVES;
      double v = 0.0;
      for (unsigned spins = 0;; ++spins) {
        bool mine = true;
        double t = 0.0;
        if (lane < NS) {
#pragma unroll 4
          for (int q = q0; q < q1; ++q) {
            const unsigned long long* w = buf + ((size_t)q * NS + lane) * 2;
            const unsigned long long lo = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long hi = __hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            mine = mine && (unsigned)(lo >> 32) == tag && (unsigned)(hi >> 32) == tag;
            t += __longlong_as_double((long long)((hi << 32) | (lo & 0xFFFFFFFFull)));
          }
        }
        if (__all(mine)) {
          v = t;
          break;
        }
        if (spins >= a.spinMax) {
          if (lane == 0) failed = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      if (lane < NS) sh[wave][lane] = v;
      __syncthreads();
      if (failed) break;  // uniform over the block
      if (tid < NS) S[tid] = ((sh[0][tid] + sh[1][tid]) + sh[2][tid]) + sh[3][tid];
      ++gen;
      __syncthreads();
    }
    if (tid < 64) {
      int next = 0;
      if (KIND == LSDG_JOB_SIM3) lm_step_sim3(s, jd, S, sP, &next, nullptr);
      else lm_step_se3(s, jd, S, sP, &next, nullptr);
    }
    __syncthreads();
  }
  if (part == 0) {
    if (tid == 0 && failed) s.status = -1;
    __syncthreads();
    block_copy(a.out, &s, TRACK_LM_BS);
  }
}

__global__ __launch_bounds__(256) void k_fill_words(unsigned long long* words, size_t n, unsigned long long value) {
  for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) words[i] = value;
}

int track_lm_blocks(lsdg_ctx c, int pixels) {
  // An evaluation shortens with the blocks, an exchange grows with them: the
  // best number goes with the square root of the points.  Measured per
  // alignment (FP32): 320x240 162 us with 16 blocks, 168 with 32, 187 with 64;
  // 640x480 175, 171, 187; 1280x960 224, 179, 172; 1920x1080 (FP16) 292, 210,
  // 189.  Alignments down to a level of up to 1.5 Mpixel keep to 64 (the finest
  // level 1280x960, SE3: 274 us, with 123 blocks 296); past it the finest level
  // outweighs the exchanges of the coarser ones (finest level 1920x1080, SE3 /
  // Sim3: 324 / 598 us with 64, 288 / 473 with 128, 299 / 472 with 160;
  // 2048x1536: 286 / 478, 218 / 328, with 200 227 / 309; 4096x3072: 648 / 1742,
  // 410 / 989, with 256 348 / 670).  The size alone decides, so that an image's
  // result does not depend on whether the host knows the count of points yet.
  const bool large = pixels > 3 << 19;
  const int nb = ((int)(std::sqrt((double)pixels) / (large ? 11.0 : 9.0)) + 4) / 8 * 8;
  return std::max(1, std::min(std::max(nb, 8), std::min(large ? TRACK_LM_MAX_BLOCKS : 64, c->num_cus)));
}

template <int KIND, int PREC>
static void (*track_kernel(int acc))(TrackLmArgs) {
  return acc == BATCH_ACC_KAHAN ? k_track_lm<KIND, PREC, ACC_TWOSUM> : k_track_lm<KIND, PREC, ACC_F64>;
}

hipError_t launch_track_lm(const TrackLmArgs& a, int prec, int acc, hipStream_t s, const KTimer* t) {
  auto k = a.jd.kind == LSDG_JOB_SIM3 ? (prec == LSDG_FP16   ? track_kernel<LSDG_JOB_SIM3, LSDG_FP16>(acc)
                                         : prec == LSDG_BF16 ? track_kernel<LSDG_JOB_SIM3, LSDG_BF16>(acc)
                                                             : track_kernel<LSDG_JOB_SIM3, LSDG_FP32>(acc))
                                      : (prec == LSDG_FP16   ? track_kernel<LSDG_JOB_SE3, LSDG_FP16>(acc)
                                         : prec == LSDG_BF16 ? track_kernel<LSDG_JOB_SE3, LSDG_BF16>(acc)
                                                             : track_kernel<LSDG_JOB_SE3, LSDG_FP32>(acc));
  return launch_k(k, dim3(a.blocks), dim3(TRACK_LM_BS), s, t, a);
}

hipError_t launch_fill_words(void* words, size_t n, unsigned long long value, hipStream_t s) {
  k_fill_words<<<dim3((unsigned)std::min<size_t>((n + 255) / 256, 256)), dim3(256), 0, s>>>(
      (unsigned long long*)words, n, value);
  return hipGetLastError();
}

}  // namespace lsdg
