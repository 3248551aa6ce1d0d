// Batched tracking: many frame-vs-keyframe alignments of uneven size, with no
// host round trip between LM iterations.  Three schedules share the LM code:
// the cooperative kernel (k_batch_coop, further down: several blocks per job,
// every level in one launch) and the two below.
//
// Whole-job kernel (k_batch_job).  While a job's level is small, one block
// runs the job's LM loop by itself: evaluation over the level's points,
// deterministic block reduction, LM step on wave 0, repeat.  No launch and no
// inter-block communication per iteration.
//
// Multi-block steps (k_batch_eval + k_batch_solve).  For larger levels each
// step is two launches.  Each job's points are cut into tiles of
// TILE = 256 * ppt points; k_batch_eval's persistent grid walks the
// concatenated tile list of all active jobs (the per-job tile counts are
// double-buffered per step so every block sees the same list) and writes each
// tile's FP64 partial sums to a fixed slot.  k_batch_solve then merges each
// job's slots in a fixed order (deterministic) and runs the job's LM step in
// one wave: the reference's accept / reject / lambda / convergence logic
// (SE3Tracker::trackFrame, Sim3Tracker::trackFrameSim3), an FP64 LDL^T solve
// and exp(d) * T, and writes the pose the job's next evaluation uses.  The
// kernel boundary between the two orders the partial sums, so no block waits
// on or fences for another.  A hipGraph replays K such steps.
#include "lm_device.h"
#include "track_device.h"

namespace lsdg {

constexpr int BATCH_BS = 256;
constexpr int BATCH_WAVES = BATCH_BS / 64;
#ifndef LSDG_BATCH_U
#define LSDG_BATCH_U 2
#endif
constexpr int BATCH_U = LSDG_BATCH_U;  // points per thread with loads in flight together
constexpr int BATCH_SOLVE_BS = 256;
constexpr int COOP_MAX_BS = 512;
// Waves per SIMD the cooperative kernel is compiled for (168 registers).  With
// two (215 registers) the loop over the points waited for memory and for the
// one wave of a block that runs the LM step: 64 Sim3 jobs of 1920x1080 1322 us,
// with three 1150.  The job's level and pose in scalar registers, counts in one
// register each, affine statistics only where they are estimated and the LM
// step's coefficients out of the loop's registers make room for it.  With four
// (128 registers, one point per thread in flight) 64 SE3 jobs of 640x480 gain
// 3%, 24 of 752x478 lose 5%, and Sim3 jobs stay where they are.
//   What the limit costs: SE3 forms take 150 to 168 registers and spill none to
// memory (two with FP32, the affine sums and compensated sums together); Sim3
// forms take all 168, and FP32 spills two (nine with the affine sums, twelve
// with compensated sums as well), FP16 and BF16 one in that last form only.
// 13 to 48 scalars sit in vector lanes.  With two waves per SIMD none spilled,
// and 64 Sim3 FP32 jobs of 640x480 took 609 us where they take 512 (affine 616
// and 516, affine and compensated 736 and 629).  Blocks of 512 threads, of which
// a CU holds one, are two waves per SIMD under the same limit.
constexpr int COOP_WAVES_PER_SIMD = 3;

// ------------------------------------------------------------- kernels
// Start state of every job: T = (frameToRef_init)^-1, first level, counters
// zero.  One block, so the remaining-jobs counter can be reset first.
__global__ __launch_bounds__(256) void k_batch_init(BatchArgs a) {
  __shared__ bool clearRows;
  if (threadIdx.x == 0) {
    *a.remaining = 0;
    // the run's epoch tags the cooperative row exchange; its low 16 bits
    // never take the value 0, which the plan's rows are cleared to when it is
    // made (its epochs start behind 1) and here whenever the low bits wrap, so
    // no word left by an earlier run can carry a tag of this one
    unsigned e = *a.epoch + 1;
    if ((e & 0xFFFFu) == 0) ++e;
    *a.epoch = e;
    clearRows = (e & 0xFFFFu) == 1;
  }
  __syncthreads();
  if (clearRows && a.coopRows)
    for (size_t i = threadIdx.x; i < a.coopWords; i += blockDim.x) a.coopRows[i] = 0ull;
  for (int j = threadIdx.x; j < a.njobs; j += blockDim.x) {
    JobState s;
    int nt = 0;
    lm_begin(s, a.jobs[j], a.P, &nt, nullptr);
    a.st[j] = s;
    a.ntiles[j] = nt;  // parity 0
    a.ntiles[a.njobs + j] = 0;
    if (nt > 0) atomicAdd(a.remaining, 1);
  }
}

// Tile evaluation of one LM step: a persistent grid walks the concatenated
// tile list of this step's jobs; each tile's FP64 partial row goes to a fixed
// slot.  No cross-block communication: the merge runs in k_batch_solve.
template <int KIND, int PREC, int ACC>
__global__ __launch_bounds__(BATCH_BS) void k_batch_eval(BatchArgs a, int parity) {
  constexpr int NS = KIND == LSDG_JOB_SIM3 ? NS_SIM3 : NS_SE3;
  __shared__ int pref[MAX_BATCH_JOBS + 1];
  __shared__ int scan_tmp[BATCH_BS];
  __shared__ double sh[BATCH_WAVES][NS];
  const int tid = threadIdx.x;
  const int nj = a.njobs;
  const int* nt = a.ntiles + parity * nj;
  // exclusive prefix of this step's tile counts (chunked block scan)
  {
    const int per = (nj + BATCH_BS - 1) / BATCH_BS;
    int base = tid * per, local = 0;
    for (int k = 0; k < per; ++k)
      if (base + k < nj) local += nt[base + k];
    scan_tmp[tid] = local;
    __syncthreads();
    for (int off = 1; off < BATCH_BS; off <<= 1) {
      int v = tid >= off ? scan_tmp[tid - off] : 0;
      __syncthreads();
      scan_tmp[tid] += v;
      __syncthreads();
    }
    int run = scan_tmp[tid] - local;
    for (int k = 0; k < per; ++k)
      if (base + k < nj) {
        pref[base + k] = run;
        run += nt[base + k];
      }
    if (tid == BATCH_BS - 1) pref[nj] = scan_tmp[BATCH_BS - 1];
    __syncthreads();
  }
  const int total = pref[nj];
  const int lane = tid & 63, wave = tid >> 6;
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    int lo = 0, hi = nj - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (pref[mid] <= t) lo = mid;
      else hi = mid - 1;
    }
    const int j = lo;
    const int tile = t - pref[j];
    const JobDesc& jd = a.jobs[j];
    const JobState* st = a.st + j;
    const int lvl = st->level;
    const JobLevel L = uniform(jd.lv[lvl]);
    const Xf x = uniform(st->xf);
    TrackKParams kp = a.kp;
    kp.aff_a = st->affA;
    kp.aff_b = st->affB;
    Accum<ACC, NS> acc;
    acc.zero();
    const int tileSize = BATCH_BS * a.ppt;
    const int i0 = tile * tileSize;
    const int i1 = min(i0 + tileSize, L.pts.n);
    if (KIND == LSDG_JOB_SIM3) {
      kp.roll[0] = st->roll[0]; kp.roll[1] = st->roll[1]; kp.roll[2] = st->roll[2]; kp.roll[3] = st->roll[3];
      sim3_points<PREC, BATCH_U, SUMS_LM_AFFINE>(L.pts, i0 + tid, BATCH_BS, i1, L.img, L.fid, L.fvar, L.g, x, kp, acc);
    } else {
      uint8_t* mask = lvl == 1 ? uniform(jd.isGood) : nullptr;
      se3_points<PREC, BATCH_U, SUMS_LM_AFFINE>(L.pts, i0 + tid, BATCH_BS, i1, L.img, L.g, x, kp, mask, acc);
    }
    const double wsum = acc.wave_slot();
    if (lane < NS) sh[wave][lane] = wsum;
    __syncthreads();
    if (tid < NS)
      a.partials[((size_t)jd.slotBase + tile) * NS + tid] = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, BATCH_WAVES);
    __syncthreads();
  }
}

// Merge and LM step of one LM iteration: one block per job.  Wave w sums the
// job's tile rows w, w + 4, ... (row order within a wave), the four wave sums
// are added in wave order, and wave 0 runs the LM step on the job's
// descriptor and control block staged in LDS (their loads are issued
// alongside the row loads).  Also zeroes the next step's tile count of jobs
// that are already finished.
template <int KIND>
__global__ __launch_bounds__(BATCH_SOLVE_BS) void k_batch_solve(BatchArgs a, int parity) {
  constexpr int NS = KIND == LSDG_JOB_SIM3 ? NS_SIM3 : NS_SE3;
  constexpr int WAVES = BATCH_SOLVE_BS / 64;
  __shared__ double part[WAVES][NS];
  __shared__ double S[NS];
  __shared__ JobState sst;
  __shared__ JobDesc sjd;
  __shared__ LmParams sP;
  __shared__ int next;
  const int j = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nj = a.njobs;
  const int n = a.ntiles[parity * nj + j];
  const int slotBase = a.jobs[j].slotBase;  // loaded alongside n
  int* ntNext = a.ntiles + (1 - parity) * nj + j;
  if (n == 0) {
    if (tid == 0) *ntNext = 0;
    return;
  }
  block_copy(&sst, a.st + j, BATCH_SOLVE_BS);
  block_copy(&sjd, a.jobs + j, BATCH_SOLVE_BS);
  block_copy(&sP, &a.P, BATCH_SOLVE_BS);
  if (lane < NS) {
    const double* rows = a.partials + (size_t)slotBase * NS + lane;
    double v = 0.0;
    int k = wave;
    for (; k + 7 * WAVES < n; k += 8 * WAVES) {
      double r[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) r[u] = rows[(size_t)(k + u * WAVES) * NS];
#pragma unroll
      for (int u = 0; u < 8; ++u) v += r[u];
    }
    for (; k < n; k += WAVES) v += rows[(size_t)k * NS];
    part[wave][lane] = v;
  }
  __syncthreads();
  if (tid < NS) {
    double v = part[0][tid];
    for (int w = 1; w < WAVES; ++w) v += part[w][tid];
    S[tid] = v;
  }
  __syncthreads();
  if (tid < 64) {
    int nx = 0;
    if (KIND == LSDG_JOB_SIM3) lm_step_sim3(sst, sjd, S, sP, &nx, a.remaining);
    else lm_step_se3(sst, sjd, S, sP, &nx, a.remaining);
    if (tid == 0) next = nx;
  }
  __syncthreads();
  block_copy(a.st + j, &sst, BATCH_SOLVE_BS);
  if (tid == 0) *ntNext = next;
}


// Whole LM of one job in one block, for as long as the job's current level
// has at most a.jobMaxPoints points: the level's evaluation over the block,
// the block's deterministic reduction (wave reduce-scatter, then waves in
// order) and the LM step on wave 0, repeated with no launch and no
// inter-block communication in between.  The job's descriptor and control
// block live in LDS meanwhile.  On exit the job is finished or stands at a
// larger level, whose tile count goes to the parity-0 slot for the
// multi-block steps.
template <int KIND, int PREC, int ACC>
__global__ __launch_bounds__(BATCH_JOB_BS) void k_batch_job(BatchArgs a) {
  constexpr int NS = KIND == LSDG_JOB_SIM3 ? NS_SIM3 : NS_SE3;
  constexpr int WAVES = BATCH_JOB_BS / 64;
  __shared__ JobState s;
  __shared__ JobDesc jd;
  __shared__ LmParams sP;
  __shared__ double sh[WAVES][NS];
  __shared__ double S[NS];
  const int j = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  block_copy(&s, a.st + j, BATCH_JOB_BS);
  block_copy(&jd, a.jobs + j, BATCH_JOB_BS);
  block_copy(&sP, &a.P, BATCH_JOB_BS);
  __syncthreads();
  for (int it = 0; it < BATCH_JOB_MAX_EVALS; ++it) {
    // s and jd are read after a barrier: the exit test is uniform over the block
    if (s.status != 0) break;
    const int lvl = uniform(s.level);
    const JobLevel L = uniform(jd.lv[lvl]);
    if (L.pts.n > a.jobMaxPoints) break;
    const Xf x = uniform(s.xf);
    TrackKParams kp = a.kp;
    kp.aff_a = uniform(s.affA);
    kp.aff_b = uniform(s.affB);
    Accum<ACC, NS> acc;
    acc.zero();
    const int n = L.pts.n;
    if (KIND == LSDG_JOB_SIM3) {
      for (int k = 0; k < 4; ++k) kp.roll[k] = uniform(s.roll[k]);
      sim3_points<PREC, BATCH_U, SUMS_LM_AFFINE>(L.pts, tid, BATCH_JOB_BS, n, L.img, L.fid, L.fvar, L.g, x, kp, acc);
    } else {
      uint8_t* mask = lvl == 1 ? uniform(jd.isGood) : nullptr;
      se3_points<PREC, BATCH_U, SUMS_LM_AFFINE>(L.pts, tid, BATCH_JOB_BS, n, L.img, L.g, x, kp, mask, acc);
    }
    const double wsum = acc.wave_slot();
    if (lane < NS) sh[wave][lane] = wsum;
    __syncthreads();
    if (tid < NS) S[tid] = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, WAVES);
    __syncthreads();
    if (tid < 64) {
      int next = 0;
      if (KIND == LSDG_JOB_SIM3) lm_step_sim3(s, jd, S, sP, &next, a.remaining);
      else lm_step_se3(s, jd, S, sP, &next, a.remaining);
    }
    __syncthreads();
  }
  block_copy(a.st + j, &s, BATCH_JOB_BS);
  if (tid == 0) a.ntiles[j] = s.status == 0 ? jd.lv[s.level].ntiles : 0;
}

// Cooperative whole-LM kernel: K blocks per job (blockIdx.x = job * K + part)
// run the job's whole LM loop together, every level included.  A level of at
// most soloMax points is evaluated whole by every block of the job.  A larger
// level is cut into K contiguous point ranges: each block reduces its range
// to an FP64 row, publishes it as tagged words (device-scope stores), reads
// the K rows until every word carries this iteration's tag, and sums them in
// a fixed order.  The rows are shared out over the block's waves: one wave
// reading them all took K dependent rounds of loads per poll (16 Sim3 jobs of
// 640x480 with 16 blocks each: 205 -> 168 us per launch; 24 SE3 jobs of
// 752x478 with 10: 345 -> 301 us per run).  In both cases every block
// of the job then holds the same sums and runs the same LM step on its own
// LDS copy of the control block, so no result is broadcast; part 0 alone
// counts finished jobs and writes the control block back.  Rows are double
// buffered by iteration parity: a block can be at most one iteration ahead of
// the slowest block of its job.  The wait is bounded (a.spinMax polls): if the
// K blocks of a job cannot all be resident (the grid is sized from the
// occupancy, so this does not happen on an idle device), the blocks stop and
// set *remaining negative, which the host reports as an error.  The block
// size (256 or 512 threads) is the launch's.
#ifndef LSDG_SPIN_SLEEP
#define LSDG_SPIN_SLEEP 2
#endif

template <int KIND, int PREC, int ACC, int SUMS>
__global__ __launch_bounds__(COOP_MAX_BS, COOP_WAVES_PER_SIMD) void k_batch_coop(BatchArgs a) {
  constexpr int NS = KIND == LSDG_JOB_SIM3 ? NS_SIM3 : NS_SE3;
  constexpr int WAVES = COOP_MAX_BS / 64;  // rows of sh; those of absent waves stay zero
  const int bs = (int)blockDim.x, waves = bs / 64;
  __shared__ JobState s;
  __shared__ JobDesc jd;
  __shared__ LmParams sP;
  __shared__ double sh[WAVES][NS];
  __shared__ double S[NS];
  __shared__ int failed;
  const int K = a.coopK;
  // Blocks are dispatched round-robin over the device's XCDs.  With
  // a.xcds > 1, block b belongs to group b % xcds, and the K blocks of job j
  // all fall in group j % xcds: a job's points and taps stay in one XCD's L2.
  int j, part;
  if (a.xcds > 1) {
    const int slot = blockIdx.x / a.xcds;
    j = (slot / K) * a.xcds + (int)(blockIdx.x % a.xcds);
    part = slot % K;
  } else {
    j = blockIdx.x / K;
    part = blockIdx.x % K;
  }
  if (j >= a.njobs) return;  // padding of the last group (the whole block leaves)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int* remaining = part == 0 ? a.remaining : nullptr;
  unsigned long long* rows = a.coopRows + (size_t)j * 2 * K * NS * 2;
  const unsigned epochTag = (*a.epoch & 0xFFFFu) << 16;
  block_copy(&s, a.st + j, bs);
  block_copy(&jd, a.jobs + j, bs);
  block_copy(&sP, &a.P, bs);
  if (tid == 0) failed = 0;
  for (int i = tid; i < WAVES * NS; i += bs) (&sh[0][0])[i] = 0.0;
  __syncthreads();
  // of level cur, in scalar registers: the job's level, whether it is split,
  // and this block's points of it
  JobLevel L{};
  int cur = -1, i0 = 0, i1 = 0;
  bool split = false;
  unsigned gen = 0;  // synchronised iterations of this job so far
  for (int it = 0; it < BATCH_JOB_MAX_EVALS; ++it) {
    // s is read after a barrier: the exit test is uniform over the block
    if (s.status != 0) break;
    const int lvl = uniform(s.level);
    if (lvl != cur) {
      cur = lvl;
      L = uniform(jd.lv[lvl]);
      split = K > 1 && L.pts.n > a.soloMax;
      const PartRange r = split ? part_range(L.pts.n, part, K) : PartRange{0, L.pts.n};
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
      sim3_points<PREC, BATCH_U, SUMS>(L.pts, i0 + tid, bs, i1, L.img, L.fid, L.fvar, L.g, x, kp, acc);
    } else {
      uint8_t* mask = lvl == 1 ? uniform(jd.isGood) : nullptr;
      se3_points<PREC, BATCH_U, SUMS>(L.pts, i0 + tid, bs, i1, L.img, L.g, x, kp, mask, acc);
    }
    const double wsum = acc.wave_slot();
    if (lane < NS) sh[wave][lane] = wsum;
    __syncthreads();
    if (!split) {
      if (tid < NS) S[tid] = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, WAVES);
    } else {
      // Tagged row exchange: each value is published as two 64-bit words
      // (one 32-bit half of the FP64 value, one 32-bit tag: the run's epoch
      // and this iteration's generation), so every word tells by itself
      // whether it belongs to this iteration.  Wave 0 stores its part's row;
      // every wave then reads its share of the K rows until all their words
      // carry the tag: one round of loads after the last part's stores land,
      // with no arrival counter and no store-completion wait in between.
      unsigned long long* buf = rows + (size_t)(gen & 1) * K * NS * 2;
      const unsigned tag = epochTag | (gen & 0xFFFFu);
      if (tid < NS) {
        const double v = Accum<ACC, NS>::merge_waves(&sh[0][tid], NS, WAVES);
        const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
        unsigned long long* w = buf + ((size_t)part * NS + tid) * 2;
        const unsigned long long t64 = (unsigned long long)tag << 32;
        __hip_atomic_store(w, t64 | (bits & 0xFFFFFFFFull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 1, t64 | (bits >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();  // sh is read above and written below
      // at most spinMax polls after the first look; a wave's rows are added
      // in part order, the waves' sums in wave order
      const int q0 = K * wave / waves, q1 = K * (wave + 1) / waves;
      double v = 0.0;
      for (unsigned spins = 0;; ++spins) {
        bool mine = true;
        double t = 0.0;
        if (lane < NS) {
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
        __builtin_amdgcn_s_sleep(LSDG_SPIN_SLEEP);
      }
      if (lane < NS) sh[wave][lane] = v;
      __syncthreads();
      if (failed) {  // uniform over the block
        if (tid == 0) __hip_atomic_store(a.remaining, -(1 << 20), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
      if (tid < NS) {
        double t = sh[0][tid];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) t += sh[w][tid];
        S[tid] = t;
      }
      ++gen;
    }
    __syncthreads();
    if (tid < 64) {
      __builtin_amdgcn_s_setprio(3);
      int next = 0;
      if (KIND == LSDG_JOB_SIM3) lm_step_sim3(s, jd, S, sP, &next, remaining);
      else lm_step_se3(s, jd, S, sP, &next, remaining);
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
  }
  if (part == 0) {
    block_copy(a.st + j, &s, bs);
    if (tid == 0) a.ntiles[j] = s.status == 0 ? jd.lv[s.level].ntiles : 0;
  }
}

// ------------------------------------------------------------ launchers
template <int KIND, int PREC>
static void (*job_kernel(int acc))(BatchArgs) {
  return acc == BATCH_ACC_KAHAN ? k_batch_job<KIND, PREC, ACC_KAHAN> : k_batch_job<KIND, PREC, ACC_F64>;
}

hipError_t launch_batch_job(const BatchArgs& a, int kind, int prec, int acc, hipStream_t s, const KTimer* t) {
  auto k = kind == LSDG_JOB_SIM3 ? (prec == LSDG_FP16   ? job_kernel<LSDG_JOB_SIM3, LSDG_FP16>(acc)
                                    : prec == LSDG_BF16 ? job_kernel<LSDG_JOB_SIM3, LSDG_BF16>(acc)
                                                        : job_kernel<LSDG_JOB_SIM3, LSDG_FP32>(acc))
                                 : (prec == LSDG_FP16   ? job_kernel<LSDG_JOB_SE3, LSDG_FP16>(acc)
                                    : prec == LSDG_BF16 ? job_kernel<LSDG_JOB_SE3, LSDG_BF16>(acc)
                                                        : job_kernel<LSDG_JOB_SE3, LSDG_FP32>(acc));
  return launch_k(k, dim3(a.njobs), dim3(BATCH_JOB_BS), s, t, a);
}

template <int ACC, int SUMS>
static void (*coop_kernel_of(int kind, int prec))(BatchArgs) {
  if (kind == LSDG_JOB_SIM3)
    return prec == LSDG_FP16 ? k_batch_coop<LSDG_JOB_SIM3, LSDG_FP16, ACC, SUMS>
           : prec == LSDG_BF16 ? k_batch_coop<LSDG_JOB_SIM3, LSDG_BF16, ACC, SUMS>
                               : k_batch_coop<LSDG_JOB_SIM3, LSDG_FP32, ACC, SUMS>;
  return prec == LSDG_FP16 ? k_batch_coop<LSDG_JOB_SE3, LSDG_FP16, ACC, SUMS>
         : prec == LSDG_BF16 ? k_batch_coop<LSDG_JOB_SE3, LSDG_BF16, ACC, SUMS>
                             : k_batch_coop<LSDG_JOB_SE3, LSDG_FP32, ACC, SUMS>;
}

static void (*coop_kernel(int kind, int prec, int acc, bool affine))(BatchArgs) {
  if (acc == BATCH_ACC_KAHAN)
    return affine ? coop_kernel_of<ACC_KAHAN, SUMS_LM_AFFINE>(kind, prec) : coop_kernel_of<ACC_KAHAN, SUMS_LM>(kind, prec);
  return affine ? coop_kernel_of<ACC_F64, SUMS_LM_AFFINE>(kind, prec) : coop_kernel_of<ACC_F64, SUMS_LM>(kind, prec);
}

bool batch_coop_block_size_ok(int bs) { return bs == 256 || bs == COOP_MAX_BS; }

int batch_coop_grid(int njobs, int K, int xcds) {
  if (xcds <= 1) return njobs * K;
  return ((njobs + xcds - 1) / xcds) * xcds * K;
}

hipError_t batch_coop_capacity(int kind, int prec, int acc, bool affine, int bs, int* blocks) {
  *blocks = 0;
  if (!batch_coop_block_size_ok(bs)) return hipErrorInvalidValue;
  int dev = 0, perCU = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, coop_kernel(kind, prec, acc, affine), bs, 0);
  *blocks = e == hipSuccess ? perCU * cus : 0;
  return e;
}

hipError_t launch_batch_coop(const BatchArgs& a, int kind, int prec, int acc, int bs, hipStream_t s,
                             const KTimer* t) {
  if (!batch_coop_block_size_ok(bs)) return hipErrorInvalidValue;
  return launch_k(coop_kernel(kind, prec, acc, a.kp.aff_stats != 0), dim3(batch_coop_grid(a.njobs, a.coopK, a.xcds)), dim3(bs), s,
                  t, a);
}

hipError_t launch_batch_init(const BatchArgs& a, hipStream_t s) {
  k_batch_init<<<dim3(1), dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

template <int KIND, int PREC>
static void (*eval_kernel(int acc))(BatchArgs, int) {
  return acc == BATCH_ACC_KAHAN ? k_batch_eval<KIND, PREC, ACC_KAHAN> : k_batch_eval<KIND, PREC, ACC_F64>;
}

hipError_t launch_batch_eval(const BatchArgs& a, int kind, int prec, int acc, int parity, int grid, hipStream_t s,
                             const KTimer* t) {
  auto k = kind == LSDG_JOB_SIM3 ? (prec == LSDG_FP16   ? eval_kernel<LSDG_JOB_SIM3, LSDG_FP16>(acc)
                                    : prec == LSDG_BF16 ? eval_kernel<LSDG_JOB_SIM3, LSDG_BF16>(acc)
                                                        : eval_kernel<LSDG_JOB_SIM3, LSDG_FP32>(acc))
                                 : (prec == LSDG_FP16   ? eval_kernel<LSDG_JOB_SE3, LSDG_FP16>(acc)
                                    : prec == LSDG_BF16 ? eval_kernel<LSDG_JOB_SE3, LSDG_BF16>(acc)
                                                        : eval_kernel<LSDG_JOB_SE3, LSDG_FP32>(acc));
  return launch_k(k, dim3(grid), dim3(BATCH_BS), s, t, a, parity);
}

hipError_t launch_batch_solve(const BatchArgs& a, int kind, int parity, hipStream_t s, const KTimer* t) {
  auto k = kind == LSDG_JOB_SIM3 ? k_batch_solve<LSDG_JOB_SIM3> : k_batch_solve<LSDG_JOB_SE3>;
  return launch_k(k, dim3(a.njobs), dim3(BATCH_SOLVE_BS), s, t, a, parity);
}

hipError_t launch_batch_step(const BatchArgs& a, int kind, int prec, int acc, int parity, int grid, hipStream_t s) {
  hipError_t e = launch_batch_eval(a, kind, prec, acc, parity, grid, s);
  if (e != hipSuccess) return e;
  return launch_batch_solve(a, kind, parity, s);
}

}  // namespace lsdg
