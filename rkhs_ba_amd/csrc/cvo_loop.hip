// The iteration loop of a registration as one resident kernel.
//
// Every block keeps its share of the source rows in LDS for the whole launch
// and runs all iterations: association of its rows, step terms of its pairs,
// controller.  Blocks meet twice an iteration, in an exchange of their partial
// sums; each block then adds all partials in the same order and runs the
// controller itself, so all blocks hold the same state and no block waits for
// a broadcast.  What bounds the launch-per-pass loop at small and middle sizes
// is not work but the chain of kernel starts, state reads and completion
// counters; here an iteration has two exchanges (2.5 us each at 256 blocks, skew of
// the blocks included).  Measured per registration, launch-per-pass loop to this
// one: 1.1k points without colour, 500 iterations 16.3 -> 9.3 ms; 5k with colour,
// 2000 iterations 60.0 -> 35.1; 60k with colour and 19 classes, 2000 iterations
// 111.6 -> 82.3; K nearest at 20k, 600 iterations 29.9 -> 24.5; adaptive
// lengthscale at 5k 7.9 -> 6.9.
//
// Exchange: a block stores its partials as 8-byte words {payload, tag} with
// device-scope stores (tag: the iteration), and its readers read all words with
// device-scope loads until the tags match: a word is its own flag, so one round
// trip carries data and arrival.  Up to 32 blocks read each other; more are
// split by XCD (block id % 8), the first block of each group sums its group and
// publishes the group's words, and every block reads the eight groups.  One
// wave per block takes part: at 256 blocks an exchange among all (32 KB read by
// every block) measured 2.1 to 2.4 us in isolation and 4.0 in the loop, where
// sixteen waves a block poll and add; two levels 1.8 in isolation and 2.5 in the
// loop; 32 blocks in one level 1.2 in isolation.
// A block can only publish iteration i + 1 of one exchange after it has read
// iteration i of the other, which every block published after reading iteration
// i of the first: one buffer per exchange and level is enough.
//
// All blocks must be resident at once: one block fits a compute unit, the host
// keeps the blocks of all such launches of the process within the device's
// compute units (a launch beside other calls has its share of them, and gives them
// back every few milliseconds), and every wait is bounded by a clock: a launch
// whose wait runs out leaves the state as it was, and the caller goes on with the
// launch-per-pass loop.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>

#include "cvo_assoc.h"
#include "cvo_controller.h"
#include "cvo_exchange.h"
#include "cvo_loop.h"

namespace cvo {

constexpr int kLoopThreads = 1024;
constexpr int kLoopWaves = kLoopThreads / 64;
constexpr int kLoopMaxBlocks = 256;
constexpr int kGroupBlocks = kLoopMaxBlocks / 8;  // blocks of an exchange's first level
constexpr uint32_t kCapped = 0x80000000u;  // a row over its cap, to be redone
// Lanes a row of the K-nearest association, whatever the tuning: at 8 the
// histograms of the rows in flight (a kilobyte each) would take the 128 KB that
// the rows need too.
constexpr int kKnnLanes = 16;

// Rows go to blocks in chunks of kChunk consecutive (Morton-sorted) rows dealt
// round robin: a block's rows come from all over its XCD's range, so dense and
// empty parts of a scene spread over the blocks (one contiguous range a block
// left the blocks waiting 20 of 53 us for the slowest, 60k street at 0.5 m).
constexpr int kChunk = 8;

// Words a block publishes after the association: the registration's six flow
// sums and, with self problems, every problem's ip sum, two words a double; then
// the stored pairs of each problem and the registration's longest row.
template <int NP>
struct AssocWords {
  static constexpr int kDoubles = NP == 1 ? 6 : 6 + NP;
  static constexpr int kCounts = NP + 1;
  static constexpr int kCount0 = 2 * kDoubles, kMaxRow = kCount0 + NP;
  static constexpr int kUsed = kMaxRow + 1;
  static constexpr int kStride = NP == 1 ? 16 : 32;
  static_assert(kUsed <= kStride, "the words exceed their line");
};
constexpr int kStepWords = 8;  // B, C, D, E

// Groups of blocks that share a contiguous range of chunks: the eight XCDs
// (block id % 8) when the blocks fill them evenly.
__host__ __device__ inline int loop_row_groups(int blocks, int xcd_remap) {
  return xcd_remap && blocks % 8 == 0 ? 8 : 1;
}

// The state's maps from LDS into scalar registers (the same for the whole block).
// SRC: the rows may be moved by a source map (the self problem of the target).
template <bool SRC>
__device__ __forceinline__ void uniform_maps(const ProblemState& s, Maps& m) {
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    m.A[i] = uni(s.A[i]);
    m.Rq[i] = uni(s.Rq[i]);
    m.As[i] = SRC ? uni(s.As[i]) : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    m.b[i] = uni(s.b[i]);
    m.Tq[i] = uni(s.Tq[i]);
    m.bs[i] = SRC ? uni(s.bs[i]) : 0.0f;
  }
  m.src_xf = SRC && uni(s.has_src_xf) != 0;
}
__device__ __forceinline__ void put_word(uint64_t* p, uint32_t payload, uint32_t tag) {
  __hip_atomic_store(p, ((uint64_t)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The wave that reads an exchange's words (read_words).
template <int PER>
struct ExchangeWave {
  static constexpr int kWords = PER;
  uint64_t v[PER];
  template <class F>
  __device__ __forceinline__ void each(F f) {
    f((int)(threadIdx.x & 63), v);
  }
  template <class F>
  __device__ __forceinline__ bool every(F f) {
    return __all(f((int)(threadIdx.x & 63), v)) != 0;
  }
};

// One wave reads the n lines of NW words at base until every tag matches and
// returns the sum over the lines of this lane's word (lane & (NW - 1)): a
// double's two words both return the double's sum, a count's word its sum, the
// word max_word its maximum.  ok is cleared, in all lanes, when the wait runs out.
template <int NW, int USED, int DOUBLE_WORDS, int LINES>
__device__ __forceinline__ double read_lines(uint64_t* base, int n_lines, uint32_t tag, uint64_t wait_ticks,
                                             int max_word, bool& ok) {
  constexpr int PER = (LINES * NW + 63) / 64;
  const int lane = threadIdx.x & 63, w = lane & (NW - 1);
  ExchangeWave<PER> wave;
  ok = read_words<NW, USED>(
           wave, n_lines, tag, wait_ticks,
           [&](int i) { return __hip_atomic_load(base + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
           []() { return (uint64_t)wall_clock64(); }) &&
       ok;
  const uint64_t(&v)[PER] = wave.v;
  double x = 0.0;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const uint32_t own = (uint32_t)v[u], other = xor_lane<1>(own);
    const uint64_t lo = (w & 1) ? other : own, hi = (w & 1) ? own : other;
    const double d = w < DOUBLE_WORDS ? __longlong_as_double((long long)((hi << 32) | lo)) : (double)own;
    x = w == max_word ? fmax(x, d) : x + d;
  }
  auto join = [&](double y) { x = w == max_word ? fmax(x, y) : x + y; };
  if constexpr (NW <= 8) join(xor_lane<8>(x));
  if constexpr (NW <= 16) join(xor_lane<16>(x));
  if constexpr (NW <= 32) join(xor_lane<32>(x));
  return x;
}

// The exchange by one wave of every block.  mine: lane w < USED the block's
// word w (a double's two words from two lanes).  Returns the totals over all
// blocks by word, as read_lines.
template <int NW, int USED, int DOUBLE_WORDS>
__device__ __forceinline__ double exchange(uint64_t* words, uint32_t mine, int n_blocks, uint32_t tag,
                                           uint64_t wait_ticks, int max_word, bool& ok) {
  const int lane = threadIdx.x & 63, b = (int)blockIdx.x;
  if (n_blocks <= kGroupBlocks) {
    if (lane < USED) put_word(words + b * NW + lane, mine, tag);
    return read_lines<NW, USED, DOUBLE_WORDS, kGroupBlocks>(words, n_blocks, tag, wait_ticks, max_word, ok);
  }
  const int grp = b & 7, member = b >> 3;
  uint64_t* line0 = words + grp * kGroupBlocks * NW;
  uint64_t* sums = words + kLoopMaxBlocks * NW;
  if (lane < USED) put_word(line0 + member * NW + lane, mine, tag);
  if (member == 0) {
    const double x = read_lines<NW, USED, DOUBLE_WORDS, kGroupBlocks>(line0, n_blocks >> 3, tag, wait_ticks, max_word, ok);
    const uint64_t bits = (uint64_t)__double_as_longlong(x);
    const uint32_t word = lane < DOUBLE_WORDS ? (uint32_t)((lane & 1) ? bits >> 32 : bits) : (uint32_t)x;
    // a wait that ran out publishes nothing: the other blocks run out too
    if (!ok) return 0.0;
    if (lane < USED) put_word(sums + grp * NW + lane, word, tag);
  }
  return read_lines<NW, USED, DOUBLE_WORDS, 8>(sums, 8, tag, wait_ticks, max_word, ok);
}

// Lane l's value of a double (l uniform).
__device__ __forceinline__ double lane_f64(double v, int l) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// One exchange of the butterfly below: the lanes with bit O keep b, the others
// a, and each gets its partner's share of what it keeps.
template <int O>
__device__ __forceinline__ double fold(double a, double b) {
  const bool up = (threadIdx.x & O) != 0;
  const double keep = up ? b : a, give = up ? a : b;
  return keep + xor_lane<O>(give);
}

// Sums of N <= 8 values over the wave: a butterfly that halves the values a
// lane carries while it doubles the lanes that share one (10 exchanges in
// place of 6 N).  Lane 8 c returns the sum of value c.
template <int N>
__device__ __forceinline__ double wave_sums(const double (&v)[N]) {
  static_assert(N == 4 || N == 6 || N == 8, "value count");
  double y0, y1;
  if constexpr (N == 4) {
    // both half waves carry the four values
    double x0 = v[0], x1 = v[1], x2 = v[2], x3 = v[3];
    x0 += xor_lane<32>(x0);
    x1 += xor_lane<32>(x1);
    x2 += xor_lane<32>(x2);
    x3 += xor_lane<32>(x3);
    y0 = fold<16>(x0, x2);
    y1 = fold<16>(x1, x3);
  } else {
    double x6 = 0.0, x7 = 0.0;
    if constexpr (N == 8) {
      x6 = v[6];
      x7 = v[7];
    }
    const double z0 = fold<32>(v[0], v[4]), z1 = fold<32>(v[1], v[5]);
    const double z2 = fold<32>(v[2], x6), z3 = fold<32>(v[3], x7);
    y0 = fold<16>(z0, z2);
    y1 = fold<16>(z1, z3);
  }
  double x = fold<8>(y0, y1);
  x += xor_lane<4>(x);
  x += xor_lane<2>(x);
  x += xor_lane<1>(x);
  return x;
}

template <int NP>
struct LoopShared {
  ProblemState st[NP];
  GridLevel lv[NP][kMaxLevels];
  float level_h[NP][kMaxLevels];
  int n_levels[NP];
  double red[kLoopWaves][9];
  double capped[kLoopWaves][7];  // a wave's sums over its capped rows
  uint32_t counts[NP + 1];       // stored pairs per problem, longest row
  float dir[6];                  // the flow's direction, for the step terms
  double xi[6], norm;            // the normalised flow and the flow's norm
  uint64_t nnz;                  // totals of the association
  uint32_t max_row;
  float rows_ell;  // lengthscale of the rows' constants
  float ind;       // the step's indicator value and decision, the next row cap
  int decay, next_K;
  int any_capped, bad;
};
template <int NP>
using SharedPtr = __attribute__((address_space(3))) LoopShared<NP>*;

// The waves' partial sums of an association to LDS.
template <int NP>
__device__ __forceinline__ void block_partials(LoopShared<NP>& S, const double (&sums)[AssocWords<NP>::kDoubles],
                                               const uint32_t (&nz)[NP], uint32_t mx) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (NP == 1) {
    const double x = wave_sums(sums);
    if ((lane & 7) == 0 && lane < 48) S.red[wave][lane >> 3] = x;
  } else {
    const double lo[8] = {sums[0], sums[1], sums[2], sums[3], sums[4], sums[5], sums[6], sums[7]};
    const double x = wave_sums(lo);
    if ((lane & 7) == 0) S.red[wave][lane >> 3] = x;
    double v = sums[8];
    v += xor_lane<32>(v);
    v += xor_lane<16>(v);
    v += xor_lane<8>(v);
    v += xor_lane<4>(v);
    v += xor_lane<2>(v);
    v += xor_lane<1>(v);
    if (lane == 0) S.red[wave][8] = v;
  }
  // integer sums: any order
#pragma unroll
  for (int q = 0; q < NP; ++q)
    if (nz[q]) atomicAdd(&S.counts[q], nz[q]);
  if (mx) atomicMax(&S.counts[NP], mx);
}

// A block's rows in LDS.
struct RowLds {
  float4* pos;
  float4* consts;  // RowConsts at LoopShared::rows_ell
  uint32_t* row;   // the row's index in its problem, ~0 for padding
  uint32_t* cnt;   // stored pairs, kCapped
  float* feat;
  float* sem;
  uint32_t* hist;
};

// Association of the block's rows [lo, hi) (local indices) of one problem, G
// lanes a row.  Adds to acc, the stored pairs to nz, the longest row to mx;
// a row over its cap is marked instead.
template <int FC, int KC, bool KNN, int G>
__device__ __forceinline__ void loop_rows(const AssocProblem& P, const KConsts& kc, const GridLevel& GL,
                                          const Maps& mp, int mode, float ell, int K, int lo, int hi, const RowLds& R,
                                          int* any_capped, double acc[7], uint32_t& nz, uint32_t& mx) {
  const int tid = threadIdx.x, g = tid & (G - 1), grp = tid / G;
  const int F = Dim<FC>::get(kc.F), KS = Dim<KC>::get(kc.Ks);
  const ExactK ek = exact_consts(kc);
  for (int i = lo + grp; i < hi; i += kLoopThreads / G) {
    const uint32_t r = R.row[i];
    if (r == ~0u) continue;
    RowResult res;
    const float4 x4 = R.pos[i], c4 = R.consts[i];
    const RowConsts rc{c4.x, c4.y, c4.z, c4.w};
    if constexpr (KNN)
      knn_row<FC, KC, G>(P, kc, ek, GL, mp, (int)r, g, mode, ell, K, x4, R.feat + i * F, R.sem + i * KS,
                         R.hist + grp * 256, res, &rc);
    else
      assoc_row<FC, KC, G, true>(P, kc, ek, GL, mp, (int)r, g, mode, ell, K, x4, R.feat + i * F, R.sem + i * KS, res,
                                 &rc);
    if (!res.overflow) {
#pragma unroll
      for (int c = 0; c < 7; ++c) acc[c] += res.acc[c];
    }
    if (g == 0) {
      R.cnt[i] = res.overflow ? kCapped : res.stored;
      if (res.overflow) *any_capped = 1;
      else {
        nz += res.stored;
        mx = max(mx, res.stored);
      }
    }
  }
}

// The launch's arguments lie in memory, read with scalar loads.  fresh() hides
// where the pointer came from, so that what a phase reads and derives from them
// is not moved out of the iteration loop: kept across the loop it would take
// several hundred registers more than a thread has (300 spilled scalar and 260
// vector registers, against none).
typedef const __attribute__((address_space(4))) LoopArgs* ArgsPtr;
__device__ __forceinline__ const LoopArgs& fresh(ArgsPtr p) {
  asm volatile("" : "+s"(p));
  return *(const LoopArgs*)p;
}

// The controller step on the shared state, by one thread: the adaptive
// lengthscale and the reference's float pose.  A call of its own: inlined, its
// FP64 temporaries would be spilled around every other phase.
template <int NP>
static __device__ __noinline__ void loop_controller_scalar(SharedPtr<NP> sp, ArgsPtr ap, bool first_block) {
  LoopShared<NP>& S = *(LoopShared<NP>*)sp;
  const LoopArgs& A = *(const LoopArgs*)(ArgsPtr)uni((const LoopArgs*)ap);
  cvo_iter_record* trace = first_block ? A.prob[0].trace : nullptr;
  if constexpr (NP > 1) {
    controller_adaptive(&S.st[0], &S.st[1], &S.st[2], A.kc, trace, A.prob[0].trace_cap, S.level_h[0], S.n_levels[0]);
#pragma unroll
    for (int q = 1; q < NP; ++q) adaptive_follow(&S.st[q], &S.st[0], q, A.kc, S.level_h[q], S.n_levels[q]);
  } else {
    controller(&S.st[0], A.kc, trace, A.prob[0].trace_cap, A.prob[0].n_src, S.level_h[0], S.n_levels[0]);
  }
}

// The part of a controller step that follows from the association's totals
// alone: the indicator windows and the next row cap (controller()).  One
// thread, while the step terms travel.
template <int NP>
static __device__ __noinline__ void loop_side(SharedPtr<NP> sp, ArgsPtr ap) {
  LoopShared<NP>& S = *(LoopShared<NP>*)sp;
  const LoopArgs& A = *(const LoopArgs*)(ArgsPtr)uni((const LoopArgs*)ap);
  const KConsts& kc = A.kc;
  if (kc.mirror_pose) return;  // the scalar controller does it all
  const uint64_t nnz = S.nnz;
  const uint32_t max_row = S.max_row;
  S.ind = (float)((double)nnz / sqrt((double)kc.n_src_f * (double)kc.n_tgt_f));
  S.decay = indicator_update(&S.st[0], S.ind, kc.window, kc.ind_thr) ? 1 : 0;
  if (kc.knn > 0) {
    const int mean = (int)ceil((double)nnz / (double)A.prob[0].n_src);
    S.next_K = min(kKnnMaxK, mean * kc.knn);
  } else {
    S.next_K = max(1, min(kc.nn_max, (int)((double)max_row * 1.2)));
  }
}

// W(i, j) of the hat matrix of p.
__device__ __forceinline__ double hat(double p0, double p1, double p2, int i, int j) {
  const int k = 3 - i - j;
  const double v = k == 0 ? p0 : (k == 1 ? p1 : p2);
  return i == j ? 0.0 : ((j - i + 3) % 3 == 1 ? -v : v);
}

// The rest of a controller step (controller()) by wave 0 with the same
// operations on the same values, spread over lanes where they are independent:
// divisions, the cubic's three roots, the entries of the 3x3 products.  One
// thread alone takes 5.5 us of dependent FP64 and LDS accesses, this 3.0 us.
template <int NP>
static __device__ __noinline__ void loop_controller_wave(SharedPtr<NP> sp, ArgsPtr ap, bool first_block) {
  LoopShared<NP>& S = *(LoopShared<NP>*)sp;
  const LoopArgs& A = *(const LoopArgs*)(ArgsPtr)uni((const LoopArgs*)ap);
  const KConsts& kc = A.kc;
  ProblemState& st = S.st[0];
  const int lane = threadIdx.x & 63;
  const int r = lane < 9 ? lane / 3 : 0, c = lane < 9 ? lane - 3 * (lane / 3) : 0;
  // state that the end needs, read early
  const double Rr0 = st.R[r * 3], Rr1 = st.R[r * 3 + 1], Rr2 = st.R[r * 3 + 2], Tr = st.T[r];
  const int k = st.iter;
  const float ell0 = st.ell;
  const float hl = S.level_h[0][min(lane, kMaxLevels - 1)];
  const int n_levels = S.n_levels[0];
  const double x0 = S.xi[0], x1 = S.xi[1], x2 = S.xi[2], x3 = S.xi[3], x4 = S.xi[4], x5 = S.xi[5];
  const double nrm = S.norm, b0 = st.bcde[0], b1 = st.bcde[1], b2 = st.bcde[2], b3 = st.bcde[3];
  // |w|, |xi| of the step's distance and, of the float direction, |w| and |v|
  double nw, nv, wn, xn;
  {
    const float f0 = (float)x0, f1 = (float)x1, f2 = (float)x2, f3 = (float)x3, f4 = (float)x4, f5 = (float)x5;
    const double qw = (double)f0 * f0 + (double)f1 * f1 + (double)f2 * f2;
    const double qv = (double)f3 * f3 + (double)f4 * f4 + (double)f5 * f5;
    const double w2 = x0 * x0 + x1 * x1 + x2 * x2;
    const double n2 = x0 * x0 + x1 * x1 + x2 * x2 + x3 * x3 + x4 * x4 + x5 * x5;
    const double q = sqrt(lane == 0 ? qw : (lane == 1 ? qv : (lane == 2 ? w2 : n2)));
    nw = lane_f64(q, 0);
    nv = lane_f64(q, 1);
    wn = lane_f64(q, 2);
    xn = lane_f64(q, 3);
  }
  cvo_iter_record rec;
  rec.ell = ell0;
  rec.nnz = (int32_t)st.nnz;
  rec.max_row = (int32_t)st.max_row;
  rec.num_neighbors = st.K;
  rec.flow_norm = (float)nrm;
  rec.step = 0.0f;
  rec.dist = 0.0f;
  rec.ip = S.ind;
  cvo_iter_record* trace = first_block && k < A.prob[0].trace_cap ? A.prob[0].trace : nullptr;
  if (nw < (double)kc.eps && nv < (double)kc.eps) {
    if (lane == 0) {
      st.ret = (nw < 1e-8 && nv < 1e-8) ? -1 : 0;
      st.done = 1;
      st.iters_out = k;
      if (trace) trace[k] = rec;
    }
    return;
  }
  // ---- step length: select_step_dev, the roots of cubic_solve by lane
  double step;
  {
    const double nan = __longlong_as_double(0x7ff8000000000000ll);
    const double a = 4.0 * b3;
    double re = nan, im = 0.0;  // lane k < 3: root k
    if (a != 0.0) {
      const double num = lane == 0 ? 3.0 * b2 : (lane == 1 ? 2.0 * b1 : b0);
      const double quo = num / a;
      const double p2 = lane_f64(quo, 0), p1 = lane_f64(quo, 1), p0 = lane_f64(quo, 2);
      if (isfinite(p2) && isfinite(p1) && isfinite(p0)) {
        const double sh = p2 / 3.0;
        const double p = p1 - p2 * sh;
        const double q = 2.0 * sh * sh * sh - sh * p1 + p0;
        const double disc = 0.25 * q * q + p * p * p / 27.0;
        double t = 0.0;
        bool refine = true;
        if (disc > 0.0) {
          const double sq = sqrt(disc);
          const double u = cbrt(-0.5 * q + (q > 0 ? -sq : sq));
          t = (u != 0.0) ? u - p / (3.0 * u) : 0.0;
          const double ci = sqrt(fmax(0.75 * t * t + p, 0.0));
          if (lane == 0) re = t - sh;
          else {
            re = -0.5 * t - sh;
            im = lane == 1 ? ci : -ci;
            refine = false;
          }
        } else if (p == 0.0) {
          re = -sh;
          refine = false;
        } else {
          const double m = 2.0 * sqrt(-p / 3.0);
          double arg = 3.0 * q / (p * m);
          arg = fmin(1.0, fmax(-1.0, arg));
          const double th = acos(arg) / 3.0;
          re = m * cos(th - 2.0943951023931954923 * (double)lane) - sh;
        }
        if (refine) {
          for (int it = 0; it < 2; ++it) {
            const double f = ((re + p2) * re + p1) * re + p0;
            const double df = (3.0 * re + 2.0 * p2) * re + p1;
            if (df == 0.0) break;
            const double ns = re - f / df;
            if (!isfinite(ns)) break;
            re = ns;
          }
        }
      }
    }
    double temp = 1.7976931348623157e308;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double ri = lane_f64(re, i), ii = lane_f64(im, i);
      if (ri > 0 && ri < temp && fabs(ii) < 1e-5) temp = ri;
    }
    step = temp;
    if (temp > (double)kc.max_step) step = (double)kc.max_step;
    else if (temp < (double)kc.min_step) step = (double)kc.min_step;
  }
  // ---- pose: R <- R dR, T <- T + R dT with (dR, dT) = se3_exp(xi, step)
  const double p0 = x0 * step, p1 = x1 * step, p2 = x2 * step;
  const double u0 = x3 * step, u1 = x4 * step, u2 = x5 * step;
  const double th2 = p0 * p0 + p1 * p1 + p2 * p2;
  const double th = sqrt(th2);
  double ca, cb, cc;
  if (th < 1e-3) {
    ca = 1.0 - th2 / 6.0 + th2 * th2 / 120.0;
    cb = 0.5 - th2 / 24.0 + th2 * th2 / 720.0;
    cc = 1.0 / 6.0 - th2 / 120.0 + th2 * th2 / 5040.0;
  } else {
    double sn, cs;
    sincos(th, &sn, &cs);
    const double num = lane == 0 ? sn : (lane == 1 ? 1.0 - cs : th - sn);
    const double den = lane == 0 ? th : (lane == 1 ? th2 : th2 * th);
    const double quo = num / den;
    ca = lane_f64(quo, 0);
    cb = lane_f64(quo, 1);
    cc = lane_f64(quo, 2);
  }
  // lane 3 r + c: entry (r, c)
  const double Wrc = hat(p0, p1, p2, r, c);
  const double w2 = hat(p0, p1, p2, r, 0) * hat(p0, p1, p2, 0, c) + hat(p0, p1, p2, r, 1) * hat(p0, p1, p2, 1, c) +
                    hat(p0, p1, p2, r, 2) * hat(p0, p1, p2, 2, c);
  const double I = r == c ? 1.0 : 0.0;
  const double dRe = I + ca * Wrc + cb * w2;
  const double Ve = I + cb * Wrc + cc * w2;
  const double pv = Ve * (c == 0 ? u0 : (c == 1 ? u1 : u2));
  const double dTr = __shfl(pv, 3 * r, 64) + __shfl(pv, 3 * r + 1, 64) + __shfl(pv, 3 * r + 2, 64);
  const double Rn = Rr0 * __shfl(dRe, c, 64) + Rr1 * __shfl(dRe, 3 + c, 64) + Rr2 * __shfl(dRe, 6 + c, 64);
  const double Tn = Tr + Rr0 * lane_f64(dTr, 0) + Rr1 * lane_f64(dTr, 3) + Rr2 * lane_f64(dTr, 6);
  double dist;
  if (step * wn < 3.0) {
    dist = step * xn;
  } else {
    double dR[9], dT[3];
#pragma unroll
    for (int i = 0; i < 9; ++i) dR[i] = lane_f64(dRe, i);
#pragma unroll
    for (int i = 0; i < 3; ++i) dT[i] = lane_f64(dTr, 3 * i);
    dist = se3_log_norm(dR, dT);
  }
  rec.step = (float)step;
  rec.dist = (float)dist;
  // ---- maps, lengthscale, shape and level of the next pass
  const double T0 = lane_f64(Tn, 0), T1 = lane_f64(Tn, 3), T2 = lane_f64(Tn, 6);
  // b(c) = -(column c of R) . T
  const double bc = -(__shfl(Rn, c, 64) * T0 + __shfl(Rn, 3 + c, 64) * T1 + __shfl(Rn, 6 + c, 64) * T2);
  if (lane < 9) {
    st.R[lane] = Rn;
    st.A[c * 3 + r] = (float)Rn;
    st.Rq[lane] = (float)Rn;
    if (c == 0) {
      st.T[r] = Tn;
      st.Tq[r] = (float)Tn;
    }
    if (r == 0) st.b[c] = (float)bc;
  }
  const bool stop = dist < (double)kc.eps_2;
  float ell = ell0;
  if (!stop && k > kc.ell_decay_start && S.decay) {
    ell = ell * kc.ell_decay_rate;
    if (ell < kc.ell_min) ell = kc.ell_min;
  }
  const bool big = policy_big(kc.pol, ell);
  const float tq = fmaxf(fabsf((float)T0), fmaxf(fabsf((float)T1), fabsf((float)T2)));
  const float need = kc.rq_coef * ell * (1.0f + kc.max_src_norm / 500.0f) * 1.0001f +
                     1e-4f * (1.0f + kc.max_src_norm + tq) + 1e-6f;
  const uint64_t fits = __ballot(lane < n_levels && hl >= need * (big ? kc.pol.scale_big : kc.pol.scale_small));
  if (lane == 0) {
    st.step = step;
    st.dist = dist;
    if (trace) trace[k] = rec;
    if (stop) {
      st.done = 1;
      st.iters_out = k;
    } else {
      st.ell = ell;
      st.K = S.next_K;
      st.iter = k + 1;
      if (k + 1 >= kc.max_iter) {
        st.done = 1;
        st.iters_out = kc.max_iter;
      }
      st.group = big ? kc.pol.group_big : kc.pol.group_small;
      st.level = fits ? 63 - __clzll((long long)fits) : 0;
      st.n_overflow = 0;
    }
  }
}

// A row over its cap, by one wave; its sums go to the wave's line of
// LoopShared::capped.  A call: rows over the cap are rare, and inlined their
// registers would be spilled in every pass.
template <int FC, int KC, int NP>
static __device__ __noinline__ uint32_t loop_capped_row(SharedPtr<NP> sp, ArgsPtr ap, int q, int r, uint32_t hist) {
  LoopShared<NP>& S = *(LoopShared<NP>*)sp;
  const LoopArgs& A = *(const LoopArgs*)(ArgsPtr)uni((const LoopArgs*)ap);
  q = uni(q);
  const AssocProblem& P = A.prob[q];
  Maps mp;
  uniform_maps<(NP > 1)>(S.st[q], mp);
  const GridLevel GL = uniform_level(S.lv[q][uni(S.st[q].level)]);
  double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const uint32_t kept = capped_row_ball<FC, KC>(P, A.kc, exact_consts(A.kc), GL, mp, uni(r), uni(S.st[q].ell),
                                                (uint32_t)uni(S.st[q].K),
                                                (uint32_t*)(__attribute__((address_space(3))) uint32_t*)hist, acc,
                                                q == 0 ? MODE_ALIGN : MODE_IP);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    double v = acc[c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) S.capped[wave][c] += v;
  }
  return kept;
}

template <int FC, int KC, bool KNN, int NP>
__global__ __launch_bounds__(kLoopThreads) void loop_kernel(const LoopArgs* args) {
  using W = AssocWords<NP>;
  ArgsPtr ap = (ArgsPtr)args;
  extern __shared__ __align__(16) char s_dyn[];
  __shared__ LoopShared<NP> S;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = gridDim.x;
  RowLds R;
  int seg[NP + 1];  // local rows of each problem: [seg[q], seg[q + 1])
  {
    const LoopArgs& A = fresh(ap);
    const KConsts& kc = A.kc;
    const int F = Dim<FC>::get(kc.F), KS = Dim<KC>::get(kc.Ks);
    R.pos = reinterpret_cast<float4*>(s_dyn);
    R.consts = R.pos + A.rows;
    R.row = reinterpret_cast<uint32_t*>(R.consts + A.rows);
    R.cnt = R.row + A.rows;
    R.feat = reinterpret_cast<float*>(R.cnt + A.rows);
    R.sem = R.feat + (FC != 0 ? A.rows * F : 0);
    R.hist = reinterpret_cast<uint32_t*>(R.sem + (KC != 0 ? A.rows * KS : 0));
    const int ng = loop_row_groups(nb, kc.xcd_remap);
    const int x = (int)blockIdx.x % ng, k = (int)blockIdx.x / ng, nbx = nb / ng;
    seg[0] = 0;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const AssocProblem& P = A.prob[q];
      const int chunks = (P.n_src + kChunk - 1) / kChunk;
      const int c0 = (int)((int64_t)chunks * x / ng), c1 = (int)((int64_t)chunks * (x + 1) / ng);
      const int mine = c1 - c0 > k ? (c1 - c0 - k + nbx - 1) / nbx : 0;
      const int lo = seg[q];
      seg[q + 1] = lo + mine * kChunk;
      for (int i = tid; i < mine * kChunk; i += kLoopThreads) {
        const int r = (c0 + k + (i / kChunk) * nbx) * kChunk + (i & (kChunk - 1));
        R.row[lo + i] = r < P.n_src ? (uint32_t)r : ~0u;
        R.cnt[lo + i] = 0u;
        R.pos[lo + i] = ld_global(P.src_pos + min(r, P.n_src - 1));
      }
      if (FC != 0)
        for (int t = tid; t < mine * kChunk * F; t += kLoopThreads) {
          const int i = t / F, f = t - i * F;
          const int r = min((c0 + k + (i / kChunk) * nbx) * kChunk + (i & (kChunk - 1)), P.n_src - 1);
          R.feat[lo * F + t] = ld_global(P.src_feat + (size_t)r * F + f);
        }
      if (KC != 0)
        for (int t = tid; t < mine * kChunk * KS; t += kLoopThreads) {
          const int i = t / KS, f = t - i * KS;
          const int r = min((c0 + k + (i / kChunk) * nbx) * kChunk + (i & (kChunk - 1)), P.n_src - 1);
          R.sem[lo * KS + t] = ld_global(P.src_sem + (size_t)r * KS + f);
        }
      const uint32_t* src = reinterpret_cast<const uint32_t*>(P.st);
      uint32_t* dst = reinterpret_cast<uint32_t*>(&S.st[q]);
      for (int t = tid; t < (int)(sizeof(ProblemState) / 4); t += kLoopThreads) dst[t] = ld_global(src + t);
      const uint32_t* gsrc = reinterpret_cast<const uint32_t*>(&P.grid->lv[0]);
      uint32_t* gdst = reinterpret_cast<uint32_t*>(&S.lv[q][0]);
      for (int t = tid; t < (int)(sizeof(GridLevel) * kMaxLevels / 4); t += kLoopThreads) gdst[t] = ld_global(gsrc + t);
      if (tid < kMaxLevels) S.level_h[q][tid] = P.grid->lv[tid].h;
      if (tid == 0) S.n_levels[q] = P.grid->n_levels;
    }
    if (tid == 0) {
      S.bad = 0;
      S.rows_ell = -1.0f;  // no lengthscale: the first iteration sets the rows' constants
      S.any_capped = 0;
    }
    if (tid < W::kCounts) S.counts[tid] = 0u;
  }
  __syncthreads();
  const int max_iters = fresh(ap).max_iters;
  for (int it = 0; it < max_iters; ++it) {
    if (S.st[0].done) break;  // uniform: every block holds the same state
    const uint32_t tag = (uint32_t)uni(S.st[0].iter) + 1u;  // never 0, and each iteration its own
    const float ell0 = uni(S.st[0].ell);
    if (ell0 != S.rows_ell) {  // uniform
      // one lengthscale for all problems; rows with their own lengthscale are
      // never moved by a source map
      const KConsts& kc = fresh(ap).kc;
      const bool own = !KNN && !kc.fixed_ell;
      for (int i = tid; i < seg[NP]; i += kLoopThreads) {
        const float4 x4 = R.pos[i];
        const RowConsts c = row_consts(kc, own, ell0, x4.x, x4.y, x4.z);
        R.consts[i] = make_float4(c.l, c.d2t, c.qg, c.r);
      }
      __syncthreads();
      if (tid == 0) S.rows_ell = ell0;
    }
    // ---- association -----------------------------------------------------
    double sums[W::kDoubles];
#pragma unroll
    for (int c = 0; c < W::kDoubles; ++c) sums[c] = 0.0;
    uint32_t nz[NP], mx = 0;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      nz[q] = 0;
      if (seg[q + 1] <= seg[q]) continue;  // uniform
      const LoopArgs& A = fresh(ap);
      const KConsts& kc = A.kc;
      const ProblemState& st = S.st[q];
      const AssocProblem& P = A.prob[q];
      Maps mp;
      uniform_maps<(NP > 1)>(st, mp);
      const GridLevel GL = uniform_level(S.lv[q][uni(st.level)]);
      const int K = uni(st.K);
      const int mode = q == 0 ? MODE_ALIGN : MODE_IP;
      double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      uint32_t mxq = 0;
      const int n = seg[q + 1] - seg[q];
#define CVO_LOOP_ROWS(G)                                                                                         \
  loop_rows<FC, KC, KNN, G>(P, kc, GL, mp, mode, ell0, K, seg[q], seg[q + 1], R, &S.any_capped, acc, nz[q], mxq)
      // As many lanes a row as one round of the block's threads holds, else 16, or 4
      // where the tuning says 4.  8 lanes are 16 here: at 60000 rows (street pair,
      // 300 iterations, cell scale 1 / 0.5) 16 took 39.7 / 31.9 ms, 4 took 59.0 /
      // 49.7, and the launch-per-pass loop at its 8 51.8 / 44.6.
      if constexpr (KNN) {
        CVO_LOOP_ROWS(kKnnLanes);
      } else {
        if (n * 64 <= kLoopThreads) CVO_LOOP_ROWS(64);
        else if (n * 32 <= kLoopThreads) CVO_LOOP_ROWS(32);
        else if (n * 16 <= kLoopThreads || uni(state_group(&st)) > 4) CVO_LOOP_ROWS(16);
        else CVO_LOOP_ROWS(4);
      }
#undef CVO_LOOP_ROWS
      if (q == 0) {
        mx = mxq;
#pragma unroll
        for (int c = 0; c < 6; ++c) sums[c] = acc[c];
      }
      if constexpr (NP > 1) sums[6 + q] = acc[6];
    }
    block_partials<NP>(S, sums, nz, mx);
    __syncthreads();
    if constexpr (!KNN) {
      if (S.any_capped) {  // uniform
        // capped rows, a wave each in turn (wave w the w-th, (w + 16)-th,
        // ...), added to the wave's partials; the mark stays until the rows'
        // next association
        uint32_t capped = 0;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          if (lane < 7) S.capped[wave][lane] = 0.0;
          for (int base = seg[q]; base < seg[q + 1]; base += 64) {
            const int i = base + lane;
            uint64_t m = __ballot(i < seg[q + 1] && (R.cnt[i] & kCapped) != 0u);
            while (m) {
              const int b = __ffsll((unsigned long long)m) - 1;
              m &= m - 1;
              if ((int)(capped % kLoopWaves) == wave) {
                const uint32_t kept = loop_capped_row<FC, KC, NP>(
                    (SharedPtr<NP>)&S, ap, q, (int)R.row[base + b],
                    (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)(R.hist + wave * 256));
                if (lane == 0) {
                  R.cnt[base + b] = kCapped | kept;
                  atomicAdd(&S.counts[q], kept);
                  if (q == 0) atomicMax(&S.counts[NP], kept);
                }
              }
              capped++;
            }
          }
          wave_lds_sync();
          if (q == 0 && lane < 6) S.red[wave][lane] += S.capped[wave][lane];
          if (NP > 1 && lane == 6) S.red[wave][6 + q] += S.capped[wave][6];
          wave_lds_sync();
        }
        __syncthreads();
      }
    }
    if (wave == 0) {
      const LoopArgs& A = fresh(ap);
      // lane w: the block's word w
      const int c = min(lane >> 1, W::kDoubles - 1);
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < kLoopWaves; ++w) v += S.red[w][c];
      const uint64_t bits = (uint64_t)__double_as_longlong(v);
      uint32_t word = (uint32_t)((lane & 1) ? bits >> 32 : bits);
      if (lane >= W::kCount0 && lane < W::kUsed) {
        word = S.counts[lane - W::kCount0];
        S.counts[lane - W::kCount0] = 0u;  // for the next association
      }
      bool ok = true;
      const double col = exchange<W::kStride, W::kUsed, 2 * W::kDoubles>(A.xa, word, nb, tag, A.wait_ticks,
                                                                         W::kMaxRow, ok);
      // lane 2 c: the scaled flow's entry c and its direction
      const double tot = col / (lane < 6 ? (double)A.kc.c : (double)A.kc.d);
      double n2 = 0.0;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const double t = lane_f64(tot, 2 * k);
        n2 += t * t;
      }
      const double nrm = sqrt(n2);
      const double xi = n2 > 0.0 ? tot / nrm : tot;
      if (lane < 12 && (lane & 1) == 0) {
        S.dir[lane >> 1] = (float)(NP > 1 ? tot : xi);
        S.st[0].flow[lane >> 1] = tot;
        S.xi[lane >> 1] = xi;
      }
      const double nnz = lane_f64(col, W::kCount0), max_row = lane_f64(col, W::kMaxRow);
      if (lane == 0) {
        S.norm = nrm;
        S.any_capped = 0;
        S.nnz = S.st[0].nnz = (uint64_t)nnz;
        S.max_row = S.st[0].max_row = (uint32_t)max_row;
        S.st[0].level_assoc = S.st[0].level;
        if (!ok) S.bad = 1;
      }
      if constexpr (NP > 1) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const double ip = lane_f64(col, 2 * (6 + q)), nzq = lane_f64(col, W::kCount0 + q);
          if (lane == 0) {
            S.st[q].ip = ip;
            S.st[q].nnz = (uint64_t)nzq;
            S.st[q].level_assoc = S.st[q].level;
          }
        }
      }
    }
    __syncthreads();
    // (a wait that ran out ends the launch after the step terms: the next
    // exchange cannot complete either)
    if (S.bad) break;  // uniform
    // ---- step terms ------------------------------------------------------
    double bcde[4] = {0.0, 0.0, 0.0, 0.0};
    {
      const LoopArgs& A = fresh(ap);
      const AssocProblem& P = A.prob[0];
      const StepDir dir{uni(S.dir[0]), uni(S.dir[1]), uni(S.dir[2]), uni(S.dir[3]), uni(S.dir[4]), uni(S.dir[5])};
      Maps mp;
      uniform_maps<false>(S.st[0], mp);
      const GridLevel GL = uniform_level(S.lv[0][uni(S.st[0].level)]);
      // lanes a row: about one for every four pairs of the mean row, within
      // the block's threads (a lane without a pair still costs its wave the
      // pair's arithmetic)
      const int rows = seg[1];
      int lsh = 0;
      while (lsh < 4 && (rows << (lsh + 1)) <= kLoopThreads && S.nnz > (uint64_t)(4 << lsh) * (uint64_t)P.n_src) ++lsh;
      const uint32_t L = 1u << lsh, l = (uint32_t)tid & (L - 1);
      for (int i = tid >> lsh; i < rows; i += kLoopThreads >> lsh) {
        const uint32_t r = R.row[i];
        if (r == ~0u) continue;
        step_row(A.kc, GL, mp, dir, R.pos[i], ell0, P.pairs + (size_t)r * P.cap_alloc, R.cnt[i] & ~kCapped, l, L, bcde);
      }
    }
    {
      const double x = wave_sums(bcde);
      if ((lane & 7) == 0 && lane < 32) S.red[wave][lane >> 3] = x;
    }
    __syncthreads();
    if (wave == 0) {
      const LoopArgs& A = fresh(ap);
      const int c = min(lane >> 1, 3);
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < kLoopWaves; ++w) v += S.red[w][c];
      const uint64_t bits = (uint64_t)__double_as_longlong(v);
      bool ok = true;
      const double x = exchange<kStepWords, kStepWords, kStepWords>(
          A.xb, (uint32_t)((lane & 1) ? bits >> 32 : bits), nb, tag, A.wait_ticks, -1, ok);
      if (lane < 8 && (lane & 1) == 0) S.st[0].bcde[lane >> 1] = x;
      if (lane == 0 && !ok) S.bad = 1;
    } else if (NP == 1 && wave == kLoopWaves - 1) {
      if (lane == 0) loop_side<NP>((SharedPtr<NP>)&S, ap);
    }
    // the controller: wave 0, with wave 15's part once that is done
    __syncthreads();
    if (S.bad) break;  // uniform
    if (wave == 0) {
      if (NP == 1 && !fresh(ap).kc.mirror_pose) loop_controller_wave<NP>((SharedPtr<NP>)&S, ap, blockIdx.x == 0);
      else if (lane == 0) loop_controller_scalar<NP>((SharedPtr<NP>)&S, ap, blockIdx.x == 0);
    }
    __syncthreads();
  }
  const LoopArgs& Ae = fresh(ap);
  if (S.bad) {
    // the state in memory stays as this launch found it
    if (tid == 0) __hip_atomic_store(Ae.flags, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  if (blockIdx.x == 0 && tid == 0) st_global(Ae.flags + 1, (uint32_t)S.st[0].done);
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const AssocProblem& P = Ae.prob[q];
    for (int i = seg[q] + tid; i < seg[q + 1]; i += kLoopThreads)
      if (R.row[i] != ~0u) st_global(P.counts + R.row[i], R.cnt[i] & ~kCapped);
    if (blockIdx.x == 0) {
      const uint32_t* src = reinterpret_cast<const uint32_t*>(&S.st[q]);
      uint32_t* dst = reinterpret_cast<uint32_t*>(P.st);
      for (int t = tid; t < (int)(sizeof(ProblemState) / 4); t += kLoopThreads) st_global(dst + t, src[t]);
    }
  }
}

// ---------------------------------------------------------------------------
// Host
// ---------------------------------------------------------------------------

// Per device, the calls of the process that use it and the compute units that its
// resident launches hold (one block a unit, whole XCD rounds: each XCD has an
// eighth of the units, and a block can only go where one is free).
struct LoopDevice {
  std::mutex mutex;
  std::condition_variable freed;
  int held = 0;
  std::atomic<int> calls{0};
};
static LoopDevice g_devices[kMaxLoopDevices];

static LoopDevice* loop_device(int dev) { return dev >= 0 && dev < kMaxLoopDevices ? &g_devices[dev] : nullptr; }

ActiveCall::ActiveCall(cvo_ctx* ctx) : ctx_(ctx) {
  LoopDevice* d = loop_device(ctx->device);
  if (ctx->call_depth++ == 0 && d) d->calls.fetch_add(1);
}
ActiveCall::~ActiveCall() {
  LoopDevice* d = loop_device(ctx_->device);
  if (--ctx_->call_depth == 0 && d) d->calls.fetch_sub(1);
}

int loop_share(int dev, int units) {
  const LoopDevice* d = loop_device(dev);
  const int calls = d ? d->calls.load() : 1;
  return calls <= 1 ? units : (units / calls) & ~7;
}

LoopUnits::~LoopUnits() {
  if (n_ == 0) return;
  LoopDevice* d = loop_device(device_);
  {
    std::lock_guard<std::mutex> lock(d->mutex);
    d->held -= n_;
  }
  d->freed.notify_all();
}
bool LoopUnits::claim(int dev, int blocks, int units, int wait_ms) {
  LoopDevice* d = loop_device(dev);
  if (!d || blocks <= 0) return false;
  const int n = std::min((blocks + 7) & ~7, units);
  std::unique_lock<std::mutex> lock(d->mutex);
  if (!d->freed.wait_for(lock, std::chrono::milliseconds(wait_ms), [&] { return d->held + n <= units; })) return false;
  d->held += n;
  device_ = dev;
  n_ = n;
  return true;
}

// The association's words (every block's line and the groups'), then the step's.
constexpr size_t kXaWords = (kLoopMaxBlocks + 8) * 32, kXbWords = (kLoopMaxBlocks + 8) * kStepWords;
size_t loop_words_bytes() { return sizeof(uint64_t) * (kXaWords + kXbWords); }
uint64_t* loop_step_words(uint64_t* words) { return words + kXaWords; }

bool loop_shape(const KConsts& kc, const int* rows, int n_probs, int units, LoopShape* out) {
  // without the distance gate every row scans all targets: that work is not
  // spread by rows
  if (!kc.use_geo || kc.uncapped || kc.mode != MODE_ALIGN || units <= 0) return false;
  // The loop saves launches, states read back and counters, about 15 us an
  // iteration; the passes have more waves in flight a row.  Registrations of 1000
  // iterations, passes / loop: planes at 60k rows 129 / 117 ms, at 80k 186 / 178,
  // street at 100k 136 / 110, at 150k 226 / 204; their first 200 iterations, which
  // have the most pairs, street at 80k 46.0 / 43.9, 120k 81.9 / 81.1, 200k 184 / 209.
  // K nearest, 600 iterations: planes at 20k 45.5 / 42.7, 30k 68.4 / 69.0, 60k 181 /
  // 196 (street at 60k 69.6 / 64.4).  Adaptive lengthscale: 15k 12.8 / 11.5, 20k 16.2 /
  // 18.7, 40k 34.0 / 41.2, from where a problem's rows take the blocks a second round.
  const int most = kc.adaptive ? 16384 : (kc.knn > 0 ? 32768 : 131072);
  int64_t total = 0;
  for (int q = 0; q < n_probs; ++q) {
    if (rows[q] > most) return false;
    total += rows[q];
  }
  if (total <= 0) return false;
  // 16 rows a block (a wave each) as far as the units go; whole XCD rounds
  int blocks = (int)std::min<int64_t>(std::min(units, kLoopMaxBlocks), (total + 15) / 16);
  if (blocks > 8) blocks &= ~7;
  const int ng = loop_row_groups(blocks, kc.xcd_remap), nbx = blocks / ng;
  LoopShape s;
  s.blocks = blocks;
  for (int q = 0; q < n_probs; ++q) {
    const int chunks = (rows[q] + kChunk - 1) / kChunk, most = (chunks + ng - 1) / ng;
    s.rows += (most + nbx - 1) / nbx * kChunk;
  }
  size_t row = 2 * sizeof(float4) + 2 * sizeof(uint32_t);
  if (kc.use_col) row += sizeof(float) * kc.F;
  if (kc.use_sem) row += sizeof(float) * kc.Ks;
  // 256-bin histograms: one per row in flight (K nearest), else one per wave
  const int hists = kc.knn > 0 ? kLoopThreads / kKnnLanes : kLoopWaves;
  s.lds = row * s.rows + sizeof(uint32_t) * 256 * (size_t)hists;
  *out = s;
  return s.lds <= kLoopMaxLds;
}

template <int FC, int KC, bool KNN, int NP>
static hipError_t launch_loop_t(const LoopArgs* a, const LoopShape& s, hipStream_t st) {
  const void* fn = reinterpret_cast<const void*>(&loop_kernel<FC, KC, KNN, NP>);
  if (s.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLoopMaxLds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((loop_kernel<FC, KC, KNN, NP>), dim3(s.blocks), dim3(kLoopThreads), s.lds, st, a);
  return hipGetLastError();
}

template <int FC, int KC>
static hipError_t launch_loop_fk(const LoopArgs* a, const KConsts& kc, const LoopShape& s, hipStream_t st) {
  if (kc.adaptive) {
    if constexpr (FC != 0) return launch_loop_t<FC, KC, false, 3>(a, s, st);
    else return hipErrorInvalidValue;  // the adaptive association always compares features
  }
  return kc.knn > 0 ? launch_loop_t<FC, KC, true, 1>(a, s, st) : launch_loop_t<FC, KC, false, 1>(a, s, st);
}

hipError_t launch_loop(const LoopArgs* a, const KConsts& kc, const LoopShape& s, hipStream_t st) {
  const int f = !kc.use_col ? 0 : (kc.F == 5 ? 5 : -1), k = !kc.use_sem ? 0 : (kc.Ks == 19 ? 19 : -1);
  if (f == 0) {
    if (k == 0) return launch_loop_fk<0, 0>(a, kc, s, st);
    if (k == 19) return launch_loop_fk<0, 19>(a, kc, s, st);
    return launch_loop_fk<0, -1>(a, kc, s, st);
  }
  if (f == 5) {
    if (k == 0) return launch_loop_fk<5, 0>(a, kc, s, st);
    if (k == 19) return launch_loop_fk<5, 19>(a, kc, s, st);
    return launch_loop_fk<5, -1>(a, kc, s, st);
  }
  if (k == 0) return launch_loop_fk<-1, 0>(a, kc, s, st);
  if (k == 19) return launch_loop_fk<-1, 19>(a, kc, s, st);
  return launch_loop_fk<-1, -1>(a, kc, s, st);
}

}  // namespace cvo
