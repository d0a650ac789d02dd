// Multi-frame IRLS bundle adjustment on the device: CvoGPU::align over frames
// and edges (src/cvo/CvoGPU.cu:1614-1671) with CvoBatchIRLS::solve
// (src/cvo/IRLS.cpp:148-367) and BinaryStateGPU (src/cvo/IRLS_State_GPU.cu:
// 144-336, src/cvo/IRLS_State_GPU.cpp:10-146).
//
// One IRLS outer iteration is one replay of a captured graph:
//   ba_prepare        per-edge maps (world transforms of both frames), cap K,
//                     grid level
//   assoc / overflow  per-edge association between the frames' world points,
//                     with per-edge stored pairs and largest row
//   ba_edges          edge on/off; stop when no edge has enough pairs
//   ba_moments        per-edge moments of the stored pairs
//   (ba_eval -> ba_assemble -> ba_solve) x (iterations_per_solve + 1)
//                     Levenberg-Marquardt over the fixed pairs
//   ba_finish         per-edge lengthscale, pose change, convergence
//
// Residuals and Jacobians are the reference's PairwiseAnalyticalDiffFunctor
// (src/cvo/IRLS_Cost_CPU.hpp:305-357): r = a |T1 p1 - T2 p2|^2 with
// J1 = diff^T dT1, J2 = -diff^T dT2 (no factor 2a), in the local
// parameterisation T <- T Exp([rho; phi]) (local_parameterization_se3.hpp:
// 21-99).  With w = P1 - P2 (world), u = [w; P1 x w] the local Jacobians are
// j1 = M1 u and j2 = -M2 u, M = [[R^T, 0], [-R^T [t]x, R^T]], so each edge only
// needs S = sum u u^T, h = sum r u and c = sum r^2 over its pairs.
//
// These are polynomials in the poses: with A = T2^-1 T1 (3x4), A0 the same at the
// poses of the association, d0 = A0 p~ - p2 (a pair's offset in frame 2 then) and
// e = (A - A0) p~, R2^T w = d = d0 + e.  So the pairs are read once an outer
// iteration, into sums over them of {1, d0, d0 d0^T}, a {1, d0, d0 d0^T, |d0|^2 d0}
// and a^2 {1, d0, d0 d0^T, |d0|^2 d0, |d0|^4} times the monomials of p1 up to the
// degree that each meets, and every candidate of the solve evaluates the
// polynomials.  p1 is taken about a mean of the edge's paired points, where the
// parts of e cancel least (about the middle of a cloud's bounding box one stray
// return at 30 km moved the poses of two outer iterations by 5e-9, one at 1000
// km, as a sensor's mark for no return, by 8e-3).  What the expansion loses is the
// cancellation of d0 against e: relative to FP64's 2e-16 a factor of
// (max(|d0|, |e|) / |d|) to the power 2 in S, 3 in h and 4 in c, none where a
// candidate moves the points by less than their offsets.  Observed: a 12-frame
// window's pose entries after 12 outer iterations against those of sums over the
// pairs at every candidate, 2e-16 of the largest.
//
// The Ceres solve is replaced by this Levenberg-Marquardt schedule:
//   D = clamp(diag(H), 1e-6, 1e32); solve (H + D/mu) d = -g;
//   rho = (F - F_new) / (-(g.d + d.H.d/2)); accept if rho > 1e-3:
//     mu /= max(1/3, 1 - (2 rho - 1)^3) (capped at 1e16), v = 2;
//   else mu /= v, v *= 2.  mu = 1e4 at the start of every solve; stop on
//   iterations_per_solve candidates, |dF|/F < 1e-5 after an accepted step,
//   ||g||inf < 1e-5 or ||d|| < 1e-5 (||x|| + 1e-5).

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "cvo_device.h"
#include "cvo_internal.h"
#include "cvo_loop.h"

namespace cvo {

constexpr int kBaMaxFrames = 64;
constexpr int kBaMaxFree = 20;                 // free frames: 120 dof, Cholesky in 115 KB of LDS
constexpr int kBaMaxDof = 6 * kBaMaxFree;
constexpr int kBaMaxEdges = 4096;
constexpr int kBaContrib = 121;                // B11, B12, B22 (36 each), g1, g2 (6 each), c
constexpr int kMomRows = 512;                  // source rows of a moment block (more where memory is short)
constexpr int kMomTiles = 5;                   // 16 x 16 tiles of the moment matrix that are used
constexpr int kMomPart = kMomTiles * 256;
constexpr int kMomUsed = 670;                  // their entries that are (mom_index)
constexpr int kSolveThreads = 256;             // four waves: the Cholesky's trailing update spread over rows
static_assert(kSolveThreads == 256 && 6 * kBaMaxFree <= kSolveThreads, "the solve's reductions assume four waves");
constexpr int kChol = 8;                       // Cholesky block: columns a panel (even, as the dof are)
constexpr int kTri = 8;                        // triangular solves: steps a load batch

struct BaEdge {
  double ell;
  int64_t nnz, nnz_last;
  int32_t f1, f2;
  int32_t K, last_max, iters_per_ell, on;
  int32_t n_rows, n_blocks;
  int32_t part0, pad;  // the first of its blocks' partials
  double centre[3];  // origin of the moments, in the source's frame (moment_origin)
};

struct BaDev {
  int32_t n_frames, n_edges, nfree, n;
  int32_t iter, done, max_iters, iters_per_solve;
  int32_t lm_iter, lm_stop, eval_pending, eval_is_candidate;
  int32_t K_init, min_nonzeros, iter_per_ell, counter_nonzero;
  int32_t stopped_no_edges, accepted_total, evals_total, h_cur;
  float ell_min_f, decay_f, rq_coef, pad_f;
  EllPolicy pol;
  double ell_min, ell_max;
  double F, Fn, mu, v, change;
  int32_t free_idx[kBaMaxFrames];
  int32_t frame_of_free[kBaMaxFree];
  float frame_norm[kBaMaxFrames];
  double X[kBaMaxFrames * 12];     // current poses, row-major 3x4 (world <- sensor)
  double Xe[kBaMaxFrames * 12];    // poses of the pending pair pass
  double Xold[kBaMaxFrames * 12];  // poses at the start of the outer iteration
  double g[kBaMaxDof], gn[kBaMaxDof], d[kBaMaxDof];
};

// ---------------------------------------------------------------------------
// Helpers
// ---------------------------------------------------------------------------

// M = [[R^T, 0], [-R^T [t]x, R^T]] of a 3x4 pose, row-major 6x6.
__device__ inline void pose_M(const double* T, double M[36]) {
  double Rt[9];
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) Rt[r * 3 + c] = T[c * 4 + r];
  const double t0 = T[3], t1 = T[7], t2 = T[11];
  const double tx[9] = {0.0, -t2, t1, t2, 0.0, -t0, -t1, t0, 0.0};
  for (int i = 0; i < 36; ++i) M[i] = 0.0;
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) {
      M[r * 6 + c] = Rt[r * 3 + c];
      M[(r + 3) * 6 + c + 3] = Rt[r * 3 + c];
      double s = 0.0;
      for (int k = 0; k < 3; ++k) s += Rt[r * 3 + k] * tx[k * 3 + c];
      M[(r + 3) * 6 + c] = -s;
    }
}

// T <- T Exp([rho; phi]), translation part first.  out may alias Tin.
__device__ inline void pose_plus(const double* Tin, const double* dlt, double* out) {
  double T[12];
  for (int i = 0; i < 12; ++i) T[i] = Tin[i];
  const double xi[6] = {dlt[3], dlt[4], dlt[5], dlt[0], dlt[1], dlt[2]};
  double dR[9], dT[3];
  se3_exp(xi, 1.0, dR, dT);
  for (int r = 0; r < 3; ++r) {
    for (int c = 0; c < 3; ++c)
      out[r * 4 + c] = T[r * 4 + 0] * dR[0 * 3 + c] + T[r * 4 + 1] * dR[1 * 3 + c] + T[r * 4 + 2] * dR[2 * 3 + c];
    out[r * 4 + 3] = T[r * 4 + 0] * dT[0] + T[r * 4 + 1] * dT[1] + T[r * 4 + 2] * dT[2] + T[r * 4 + 3];
  }
}

// Float maps of an edge: source and target world transforms, and the query
// map from the world into the target's sensor frame.
__device__ inline void edge_maps(const double* T1, const double* T2, ProblemState* st) {
  for (int r = 0; r < 3; ++r) {
    for (int c = 0; c < 3; ++c) {
      st->As[r * 3 + c] = (float)T1[r * 4 + c];
      st->A[r * 3 + c] = (float)T2[r * 4 + c];
      st->Rq[r * 3 + c] = (float)T2[c * 4 + r];
    }
    st->bs[r] = (float)T1[r * 4 + 3];
    st->b[r] = (float)T2[r * 4 + 3];
    st->Tq[r] = (float)(-(T2[0 * 4 + r] * T2[3] + T2[1 * 4 + r] * T2[7] + T2[2 * 4 + r] * T2[11]));
  }
  st->has_src_xf = 1;
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void ba_prepare_kernel(BaDev* __restrict__ ba, BaEdge* __restrict__ edges,
                                                         const AssocProblem* __restrict__ probs) {
  const int tid = threadIdx.x;
  const bool done = ba->done != 0;
  const int E = ba->n_edges;
  if (done) {
    for (int e = tid; e < E; e += blockDim.x) probs[e].st->done = 1;
    return;
  }
  for (int i = tid; i < ba->n_frames * 12; i += blockDim.x) {
    ba->Xold[i] = ba->X[i];
    ba->Xe[i] = ba->X[i];
  }
  for (int e = tid; e < E; e += blockDim.x) {
    BaEdge& ed = edges[e];
    ProblemState* st = probs[e].st;
    ed.nnz_last = ed.nnz;
    if (ed.last_max > 0) ed.K = min(ba->K_init, (int)((double)ed.last_max * 1.1));
    if (ed.K < 1) ed.K = 1;
    const double* T1 = ba->X + 12 * ed.f1;
    const double* T2 = ba->X + 12 * ed.f2;
    edge_maps(T1, T2, st);
    st->ell = (float)ed.ell;
    st->K = ed.K;
    st->iter = ba->iter;
    st->done = 0;
    st->n_overflow = 0;
    // query radius bound at this lengthscale over the world-frame source
    const double tn = sqrt(T1[3] * T1[3] + T1[7] * T1[7] + T1[11] * T1[11]);
    const float sn = ba->frame_norm[ed.f1] + (float)tn;
    const float tq = fmaxf(fabsf(st->Tq[0]), fmaxf(fabsf(st->Tq[1]), fabsf(st->Tq[2])));
    const float r_need =
        ba->rq_coef * st->ell * (1.0f + sn / 500.0f) * 1.0001f + 1e-4f * (1.0f + sn + tq) + 1e-6f;
    const bool big = policy_big(ba->pol, st->ell);
    st->group = big ? ba->pol.group_big : ba->pol.group_small;
    st->level = choose_level(probs[e].grid, r_need * (big ? ba->pol.scale_big : ba->pol.scale_small));
  }
}

// Edge switches after the association (IRLS.cpp:235-250,
// IRLS_State_GPU.cpp:17-21) and the start of the Levenberg-Marquardt solve.
__global__ __launch_bounds__(256) void ba_edges_kernel(BaDev* __restrict__ ba, BaEdge* __restrict__ edges,
                                                       const AssocProblem* __restrict__ probs) {
  if (ba->done) return;
  const int tid = threadIdx.x;
  __shared__ int s_cnt[256];
  int cnt = 0;
  for (int e = tid; e < ba->n_edges; e += blockDim.x) {
    BaEdge& ed = edges[e];
    const ProblemState* st = probs[e].st;
    ed.nnz = (int64_t)st->nnz;
    ed.last_max = (int32_t)st->max_row;
    ed.on = (ed.nnz > 0 && ed.nnz >= (int64_t)ba->min_nonzeros) ? 1 : 0;
    if (ed.nnz > (int64_t)ba->min_nonzeros) cnt++;
  }
  s_cnt[tid] = cnt;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) s_cnt[tid] += s_cnt[tid + w];
    __syncthreads();
  }
  if (tid == 0) {
    ba->counter_nonzero = s_cnt[0];
    if (s_cnt[0] == 0) {
      ba->done = 1;
      ba->stopped_no_edges = 1;
      ba->eval_pending = 0;
      return;
    }
    ba->mu = 1e4;
    ba->v = 2.0;
    ba->lm_iter = 0;
    ba->lm_stop = 0;
    ba->eval_is_candidate = 0;
    ba->eval_pending = ba->n > 0 ? 1 : 0;
  }
}

// ---------------------------------------------------------------------------
// Moments of an edge's pairs
// ---------------------------------------------------------------------------

// Monomials x^i y^j z^k of degree <= 4, by degree: 1; x, y, z; xx, xy, xz, yy,
// yz, zz; 10 of degree 3; 15 of degree 4.  The first 4 carry a linear form, the
// first 10 a quadratic one.
constexpr int kMono = 35, kQuad = 10, kLin = 4;
struct MonoTables {
  int8_t mul[kQuad][kQuad];  // index of the product of two of the first ten
  constexpr MonoTables() : mul() {
    int e[kMono][3] = {};
    int n = 0;
    for (int d = 0; d <= 4; ++d)
      for (int i = d; i >= 0; --i)
        for (int j = d - i; j >= 0; --j) {
          e[n][0] = i;
          e[n][1] = j;
          e[n][2] = d - i - j;
          ++n;
        }
    for (int a = 0; a < kQuad; ++a)
      for (int b = 0; b < kQuad; ++b)
        for (int m = 0; m < kMono; ++m)
          if (e[m][0] == e[a][0] + e[b][0] && e[m][1] == e[a][1] + e[b][1] && e[m][2] == e[a][2] + e[b][2])
            mul[a][b] = (int8_t)m;
  }
};
__constant__ MonoTables kMonoTab;

// Row moments and where their sums lie.  The moment matrix has 37 rows (a sum
// over a source row's pairs each) by 35 monomials of the row's point; rows are
// laid out so that 16 x 16 tiles hold what is used: tile row 0 the moments of
// degree 0 and 1 in d0, which meet monomials up to degree 4 (tiles 0, 1, 2), tile
// rows 1 and 2 those of degree 2 to 4, which meet degree <= 2 (tiles 3, 4).
constexpr int kM_n = 0, kM_a0 = 1, kM_b0 = 2, kM_D1 = 3, kM_a1 = 6, kM_b1 = 9;
constexpr int kM_D2 = 16, kM_a2 = 22, kM_b2 = 28, kM_a3 = 34, kM_b3 = 37, kM_b4 = 40, kMomRowsUsed = 41;

// Where an entry of the tiles lies in a stored set of moments, -1 if nothing
// uses it.  Tiles 0 to 2 have 12 rows, the last of them 3 columns; tiles 3 and 4
// have 10 columns, the last of them 9 rows.
__device__ __forceinline__ int mom_index(int i) {
  const int t = i >> 8, r = (i >> 4) & 15, c = i & 15;
  if (t < 3) return r < 12 && (t < 2 || c < kMono - 32) ? (t < 2 ? t * 192 + r * 16 + c : 384 + r * 3 + c) : -1;
  return c < kQuad && (t < 4 || r < kMomRowsUsed - 32) ? 420 + (t - 3) * 160 + r * kQuad + c : -1;
}
static_assert(kMomUsed == 2 * 12 * 16 + 12 * (kMono - 32) + 16 * kQuad + (kMomRowsUsed - 32) * kQuad, "the stored entries");
// An edge's moments lie in its slot of the association's capped-row partials,
// which the association is done with by then.
static_assert(kMomUsed <= 10 * kOvfBlocks, "the moments fit the slots");

// Sum of moment m times monomial q in the summed tiles.
__device__ __forceinline__ double mom(const double* s_m, int m, int q) {
  const int tile = m < 16 ? q >> 4 : 2 + (m >> 4);
  return s_m[tile * 256 + (m & 15) * 16 + (q & 15)];
}

// The relative map T2^-1 T1 (row-major 3x4) of two poses.
__device__ __forceinline__ void relative_map(const double* T1, const double* T2, double A[12]) {
#pragma unroll
  for (int r = 0; r < 3; ++r) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      A[r * 4 + c] = fma(T2[8 + r], T1[8 + c], fma(T2[4 + r], T1[4 + c], T2[r] * T1[c]));
    A[r * 4 + 3] = fma(T2[8 + r], T1[11] - T2[11], fma(T2[4 + r], T1[7] - T2[7], T2[r] * (T1[3] - T2[3])));
  }
}

// The origin of an edge's moments: the mean of the paired rows among 256 spread
// over the edge's rows, of the next such set where none of these has a pair.  Each
// block of the edge forms it, with the same operations; a launch of its own for the
// mean of all would add 10 us to an outer iteration.  s: 16 words of LDS.
__device__ __forceinline__ void moment_origin(const AssocProblem& P, double* s, double c[3]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int stride = (P.n_src + 255) / 256;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < stride; ++k) {
    const int r = tid * stride + k;
    if (r < P.n_src && ld_global(P.counts + r) != 0u) {
      const float4 p = ld_global(P.src_pos + r);
      v[0] = (double)p.x;
      v[1] = (double)p.y;
      v[2] = (double)p.z;
      v[3] = 1.0;
    }
    if (__syncthreads_or(v[3] != 0.0)) break;  // an edge that is on has pairs
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
    if (lane == 0) s[wave * 4 + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = ((s[k] + s[4 + k]) + s[8 + k]) + s[12 + k];
#pragma unroll
  for (int k = 0; k < 3; ++k) c[k] = uni(v[k] / v[3]);
  __syncthreads();  // s is used again
}

// The pairs' moments, once an outer iteration (at the association's poses, X).
// A lane owns a source row and reads its pairs in order, four loads in flight;
// FP64 sums of 37 moments in registers.  Then the wave's 64 rows times their
// monomials: sums over rows of products, so FP64 matrix instructions
// (v_mfma_f64_16x16x4, 16 rows of the cloud staged in LDS at a time).  Block
// partials of the five tiles' 670 used entries.  Bound by FP64 issue and the rows' uneven lengths;
// a pass over the pairs of each candidate took 187 us and 11 for its sums, nine
// times an outer iteration (window of 12 frames of 5k to 40k points), this 306 us
// once and 8.6 us for each candidate's polynomials (window: 61.7 -> 45.3 ms for 12
// outer iterations; over 60, whose rows get longer, 420 us a pass).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void ba_moments_kernel(
    const BaDev* __restrict__ ba, BaEdge* __restrict__ edges, const AssocProblem* __restrict__ probs,
    double* __restrict__ part, int rows) {
  if (ba->done || !ba->eval_pending) return;
  const int e = blockIdx.y;
  const BaEdge& ed = edges[e];
  if (!ed.on || (int)blockIdx.x >= ed.n_blocks) return;
  const AssocProblem& P = probs[e];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  typedef double double4_t __attribute__((ext_vector_type(4)));
  constexpr int kSM = 49, kSQ = 49;  // doubles a staged row of moments / monomials (odd: no bank pattern)
  __shared__ double s_stage[4][16 * (kSM + kSQ)];
  double* s_m = s_stage[wave];
  double* s_q = s_m + 16 * kSM;
  // pairs are stored at the row stride of this iteration's cap (the
  // reference re-strides its pair matrix the same way)
  const size_t row_stride = (size_t)P.st->K;
  double A[12];
  relative_map(ba->X + 12 * ed.f1, ba->X + 12 * ed.f2, A);
  double c[3];
  moment_origin(P, s_stage[0], c);
  const double c0 = c[0], c1 = c[1], c2 = c[2];
  if (blockIdx.x == 0 && tid < 3) edges[e].centre[tid] = tid == 0 ? c0 : (tid == 1 ? c1 : c2);
  double4_t acc[kMomTiles];
#pragma unroll
  for (int t = 0; t < kMomTiles; ++t) acc[t] = (double4_t){0.0, 0.0, 0.0, 0.0};
  for (int base = blockIdx.x * rows; base < (int)(blockIdx.x + 1) * rows && base < P.n_src; base += 256) {
    const int r = base + wave * 64 + lane;
    uint32_t cnt = 0;
    double y0 = 0.0, y1 = 0.0, y2 = 0.0, x = 0.0, y = 0.0, z = 0.0;
    if (r < P.n_src) {
      cnt = ld_global(P.counts + r);
      const float4 p4 = ld_global(P.src_pos + r);
      const double p0 = p4.x, p1 = p4.y, p2 = p4.z;
      y0 = fma(A[2], p2, fma(A[1], p1, fma(A[0], p0, A[3])));
      y1 = fma(A[6], p2, fma(A[5], p1, fma(A[4], p0, A[7])));
      y2 = fma(A[10], p2, fma(A[9], p1, fma(A[8], p0, A[11])));
      x = p0 - c0;
      y = p1 - c1;
      z = p2 - c2;
    }
    if (__ballot(cnt != 0) == 0ull) continue;  // the wave's rows hold no pair
    double D1[3] = {}, D2[6] = {}, a0 = 0.0, a1[3] = {}, a2[6] = {}, a3[3] = {};
    double b0 = 0.0, b1[3] = {}, b2[6] = {}, b3[3] = {}, b4 = 0.0;
    auto add = [&](const float4& q) {
      const double d[3] = {y0 - (double)q.x, y1 - (double)q.y, y2 - (double)q.z};
      const double a = (double)q.w, b = a * a;
      const double n2 = fma(d[2], d[2], fma(d[1], d[1], d[0] * d[0]));
      const double an = a * n2, bn = b * n2;
      a0 += a;
      b0 += b;
      b4 = fma(bn, n2, b4);
      int k = 0;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        D1[i] += d[i];
        a1[i] = fma(a, d[i], a1[i]);
        b1[i] = fma(b, d[i], b1[i]);
        a3[i] = fma(an, d[i], a3[i]);
        b3[i] = fma(bn, d[i], b3[i]);
#pragma unroll
        for (int j = i; j < 3; ++j) {
          const double dd = d[i] * d[j];
          D2[k] += dd;
          a2[k] = fma(a, dd, a2[k]);
          b2[k] = fma(b, dd, b2[k]);
          ++k;
        }
      }
    };
    {
      const float4* row = P.pairs4 + (size_t)r * row_stride;
      uint32_t s = 0;
      for (; s + 4 <= cnt; s += 4) {
        const float4 q0 = ld_global(row + s), q1 = ld_global(row + s + 1), q2 = ld_global(row + s + 2),
                     q3 = ld_global(row + s + 3);
        add(q0);
        add(q1);
        add(q2);
        add(q3);
      }
      for (; s < cnt; ++s) add(ld_global(row + s));
    }
#pragma unroll 1
    for (int quarter = 0; quarter < 4; ++quarter) {
      if ((lane >> 4) == quarter) {
        double* m = s_m + (lane & 15) * kSM;
        double* q = s_q + (lane & 15) * kSQ;
        m[kM_n] = (double)cnt;
        m[kM_a0] = a0;
        m[kM_b0] = b0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          m[kM_D1 + i] = D1[i];
          m[kM_a1 + i] = a1[i];
          m[kM_b1 + i] = b1[i];
          m[kM_a3 + i] = a3[i];
          m[kM_b3 + i] = b3[i];
        }
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          m[kM_D2 + i] = D2[i];
          m[kM_a2 + i] = a2[i];
          m[kM_b2 + i] = b2[i];
        }
#pragma unroll
        for (int i = 12; i < 16; ++i) m[i] = 0.0;
        m[kM_b4] = b4;
#pragma unroll
        for (int i = kMomRowsUsed; i < 48; ++i) m[i] = 0.0;
        // monomials: those of degree d from those of degree d - 1
        double v[kMono];
        v[0] = 1.0;
        v[1] = x;
        v[2] = y;
        v[3] = z;
        v[4] = x * x;
        v[5] = x * y;
        v[6] = x * z;
        v[7] = y * y;
        v[8] = y * z;
        v[9] = z * z;
#pragma unroll
        for (int i = 0; i < 6; ++i) v[10 + i] = x * v[4 + i];
#pragma unroll
        for (int i = 0; i < 3; ++i) v[16 + i] = y * v[7 + i];
        v[19] = z * v[9];
#pragma unroll
        for (int i = 0; i < 10; ++i) v[20 + i] = x * v[10 + i];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[30 + i] = y * v[16 + i];
        v[34] = z * v[19];
#pragma unroll
        for (int i = 0; i < kMono; ++i) q[i] = v[i];
#pragma unroll
        for (int i = kMono; i < 48; ++i) q[i] = 0.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int k0 = 0; k0 < 16; k0 += 4) {
        const double* m = s_m + (k0 + (lane >> 4)) * kSM + (lane & 15);
        const double* q = s_q + (k0 + (lane >> 4)) * kSQ + (lane & 15);
        const double m0 = m[0], q0 = q[0];
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0, q0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0, q[16], acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0, q[32], acc[2], 0, 0, 0);
        acc[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[16], q0, acc[3], 0, 0, 0);
        acc[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[32], q0, acc[4], 0, 0, 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  // the four waves' tiles in order; lane: rows (lane >> 4) + 4 v, column lane & 15
  double* out = part + (size_t)(ed.part0 + blockIdx.x) * kMomUsed;
  static_assert(16 * (kSM + kSQ) >= kMomPart, "a wave's tiles fit its staging");
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kMomTiles; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) s_stage[wave][t * 256 + ((lane >> 4) + 4 * v) * 16 + (lane & 15)] = acc[t][v];
  __syncthreads();
  for (int i = tid; i < kMomPart; i += 256) {
    const int k = mom_index(i);
    if (k >= 0) out[k] = ((s_stage[0][i] + s_stage[1][i]) + s_stage[2][i]) + s_stage[3][i];
  }
}

// An edge's moments: the blocks' partials in order.
__global__ __launch_bounds__(256) void ba_moments_sum_kernel(const BaDev* __restrict__ ba,
                                                             const BaEdge* __restrict__ edges,
                                                             const double* __restrict__ part,
                                                             double* __restrict__ moments) {
  if (ba->done || !ba->eval_pending) return;
  const int e = blockIdx.x;
  const BaEdge& ed = edges[e];
  if (!ed.on) return;
  const int i = blockIdx.y * 256 + threadIdx.x;
  if (i >= kMomUsed) return;
  const double* p = part + (size_t)ed.part0 * kMomUsed + i;
  double v = 0.0;
#pragma unroll 8
  for (int b = 0; b < ed.n_blocks; ++b) v += p[(size_t)b * kMomUsed];
  moments[(size_t)e * kMomUsed + i] = v;
}

// S, h and c of an edge at the poses Xe from its moments, and the edge's blocks
// of the normal equations: B11 = M1 S M1^T, B12 = -M1 S M2^T, B22 = M2 S M2^T,
// g1 = M1 h, g2 = -M2 h.  In frame 2 with u' = [d; s x d], s = A p~ + R2^T t2,
// u = diag(R2, R2) u':
//   V_ik[f] = sum f d_i d_k for f = 1, s_b, s_b s_c    (S')
//   F_i[f] = sum f a |d|^2 d_i for f = 1, s_b          (h')
// as polynomials over the monomials.  Four lanes per V and F entry (each a
// quarter of the outer sum's terms, added in order), one wave for c.
__global__ __launch_bounds__(384) void ba_eval_kernel(const BaDev* __restrict__ ba, const BaEdge* __restrict__ edges,
                                                      const double* __restrict__ moments,
                                                      double* __restrict__ contrib) {
  if (ba->done || !ba->eval_pending) return;
  const int e = blockIdx.x;
  const BaEdge& ed = edges[e];
  if (!ed.on) return;
  const int tid = threadIdx.x;
  __shared__ double s_m[kMomPart];
  __shared__ double s_e[3][kLin];        // e_i over (1, x, y, z)
  __shared__ double s_f[10][kQuad];      // 1; s_b; s_b s_c (00 01 02 11 12 22)
  __shared__ double s_ee[6][kQuad];      // e_i e_k
  __shared__ double s_g[kQuad];          // |e|^2
  __shared__ double s_fe[12][kQuad];     // f e_i, f = 1, s_b
  __shared__ double s_V[60], s_F[12], s_c;
  __shared__ int8_t s_mul[kQuad][kQuad];
  __shared__ double s_M1[36], s_M2[36], s_N1[36], s_N2[36], s_S[36], s_h[6], s_T1[36], s_T2[36];
  for (int i = tid; i < kMomPart; i += blockDim.x) {
    const int k = mom_index(i);
    s_m[i] = k >= 0 ? moments[(size_t)e * kMomUsed + k] : 0.0;
  }
  if (tid < kQuad * kQuad) s_mul[tid / kQuad][tid % kQuad] = kMonoTab.mul[tid / kQuad][tid % kQuad];
  const double* T2 = ba->Xe + 12 * ed.f2;
  if (tid == 128) pose_M(ba->Xe + 12 * ed.f1, s_M1);
  if (tid == 192) pose_M(T2, s_M2);
  if (tid < 3) {
    double A[12], A0[12];
    relative_map(ba->Xe + 12 * ed.f1, T2, A);
    relative_map(ba->Xold + 12 * ed.f1, ba->Xold + 12 * ed.f2, A0);
    const double* c = ed.centre;
    const int r = tid;
    double Ar[4], A0r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // row r, without indexing registers
      Ar[k] = r == 0 ? A[k] : (r == 1 ? A[4 + k] : A[8 + k]);
      A0r[k] = r == 0 ? A0[k] : (r == 1 ? A0[4 + k] : A0[8 + k]);
    }
    const double at = fma(Ar[2], c[2], fma(Ar[1], c[1], fma(Ar[0], c[0], Ar[3])));
    const double a0t = fma(A0r[2], c[2], fma(A0r[1], c[1], fma(A0r[0], c[0], A0r[3])));
    // (R2^T t2)_r
    const double tau = fma(T2[8 + r], T2[11], fma(T2[4 + r], T2[7], T2[r] * T2[3]));
    s_e[r][0] = at - a0t;
    s_f[1 + r][0] = at + tau;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s_e[r][1 + k] = Ar[k] - A0r[k];
      s_f[1 + r][1 + k] = Ar[k];
    }
#pragma unroll
    for (int k = kLin; k < kQuad; ++k) s_f[1 + r][k] = 0.0;
  }
  if (tid >= 64 && tid < 64 + kQuad) s_f[0][tid - 64] = tid == 64 ? 1.0 : 0.0;
  __syncthreads();
  // products of two linear forms: thread (form pair, monomial)
  if (tid < 24 * kQuad) {
    const int w = tid / kQuad, q = tid - w * kQuad;
    const double* u;
    const double* v;
    double* out;
    if (w < 12) {
      const int k = w < 6 ? w : w - 6;
      const int i = k < 3 ? 0 : (k < 5 ? 1 : 2), j = k < 3 ? k : (k < 5 ? k - 2 : 2);
      u = w < 6 ? s_e[i] : s_f[1 + i];
      v = w < 6 ? s_e[j] : s_f[1 + j];
      out = w < 6 ? s_ee[k] : s_f[4 + k];
    } else {
      u = s_f[(w - 12) / 3];
      v = s_e[(w - 12) % 3];
      out = s_fe[w - 12];
    }
    double x = 0.0;
#pragma unroll
    for (int i = 0; i < kLin; ++i)
#pragma unroll
      for (int j = 0; j < kLin; ++j)
        if (s_mul[i][j] == q) x = fma(u[i], v[j], x);
    out[q] = x;
  }
  __syncthreads();
  if (tid < kQuad) s_g[tid] = (s_ee[0][tid] + s_ee[3][tid]) + s_ee[5][tid];
  __syncthreads();
  if (tid < 240) {
    const int o = tid >> 2, part = tid & 3, f = o / 6, k = o - f * 6;
    const int i = k < 3 ? 0 : (k < 5 ? 1 : 2), j = k < 3 ? k : (k < 5 ? k - 2 : 2);
    const int nf = f == 0 ? 1 : (f < 4 ? kLin : kQuad);
    double x = 0.0;
    for (int a = part; a < nf; a += 4) {
      double y = mom(s_m, kM_D2 + k, a);
#pragma unroll
      for (int l = 0; l < kLin; ++l) {
        const int q = s_mul[a][l];
        y = fma(s_e[j][l], mom(s_m, kM_D1 + i, q), y);
        y = fma(s_e[i][l], mom(s_m, kM_D1 + j, q), y);
      }
#pragma unroll
      for (int l = 0; l < kQuad; ++l) y = fma(s_ee[k][l], mom(s_m, kM_n, s_mul[a][l]), y);
      x = fma(s_f[f][a], y, x);
    }
    const double x1 = __shfl_xor(x, 1, 64);
    x = (tid & 1) ? x1 + x : x + x1;
    const double x2 = __shfl_xor(x, 2, 64);
    x = (tid & 2) ? x2 + x : x + x2;
    if (part == 0) s_V[o] = x;
  } else if (tid >= 256 && tid < 304) {
    const int o = (tid - 256) >> 2, part = tid & 3, f = o / 3, i = o - f * 3;
    const int nf = f == 0 ? 1 : kLin;
    double x = 0.0;
    if (part < nf) {
      // f's monomial `part`: a3, a2 e, and the quadratics of e times a1
      double y = mom(s_m, kM_a3 + i, part);
#pragma unroll
      for (int l = 0; l < kLin; ++l) {
        const int q = s_mul[part][l];
        const double tr = (mom(s_m, kM_a2, q) + mom(s_m, kM_a2 + 3, q)) + mom(s_m, kM_a2 + 5, q);
        y = fma(tr, s_e[i][l], y);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int lo = min(i, k), hi = max(i, k), ik = lo == 0 ? hi : lo + hi + 1;
          y = fma(2.0 * mom(s_m, kM_a2 + ik, q), s_e[k][l], y);
        }
      }
#pragma unroll
      for (int l = 0; l < kQuad; ++l) {
        const int q = s_mul[part][l];
        y = fma(s_g[l], mom(s_m, kM_a1 + i, q), y);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int lo = min(i, k), hi = max(i, k), ik = lo == 0 ? hi : lo + hi + 1;
          y = fma(2.0 * s_ee[ik][l], mom(s_m, kM_a1 + k, q), y);
        }
      }
      x = s_f[f][part] * y;
    }
    // |e|^2 a0 (f e_i)
    for (int a = part; a < kQuad; a += 4) {
      double y = 0.0;
#pragma unroll
      for (int l = 0; l < kQuad; ++l) y = fma(s_g[l], mom(s_m, kM_a0, s_mul[a][l]), y);
      x = fma(s_fe[o][a], y, x);
    }
    const double x1 = __shfl_xor(x, 1, 64);
    x = (tid & 1) ? x1 + x : x + x1;
    const double x2 = __shfl_xor(x, 2, 64);
    x = (tid & 2) ? x2 + x : x + x2;
    if (part == 0) s_F[o] = x;
  } else if (tid >= 320) {
    // c = sum a^2 |d|^4
    const int l = tid - 320;
    double x = 0.0;
    for (int t = l; t < 1 + 12 + kQuad + 60 + 30 * kLin + 100; t += 64) {
      int k = t;
      if (k < 1) {
        x += mom(s_m, kM_b4, 0);
        continue;
      }
      k -= 1;
      if (k < 12) {  // 4 e . b3
        x = fma(4.0 * s_e[k >> 2][k & 3], mom(s_m, kM_b3 + (k >> 2), k & 3), x);
        continue;
      }
      k -= 12;
      if (k < kQuad) {  // 2 |e|^2 tr b2
        const double tr = (mom(s_m, kM_b2, k) + mom(s_m, kM_b2 + 3, k)) + mom(s_m, kM_b2 + 5, k);
        x = fma(2.0 * s_g[k], tr, x);
        continue;
      }
      k -= kQuad;
      if (k < 60) {  // 4 e^T b2 e
        const int ik = k / kQuad, q = k - ik * kQuad;
        const double w = ik == 0 || ik == 3 || ik == 5 ? 4.0 : 8.0;
        x = fma(w * s_ee[ik][q], mom(s_m, kM_b2 + ik, q), x);
        continue;
      }
      k -= 60;
      if (k < 30 * kLin) {  // 4 |e|^2 e . b1
        const int i = k / 40, a = (k - i * 40) >> 2, q = k & 3;
        x = fma(4.0 * s_g[a] * s_e[i][q], mom(s_m, kM_b1 + i, s_mul[a][q]), x);
        continue;
      }
      k -= 30 * kLin;
      const int a = k / kQuad, q = k - a * kQuad;  // |e|^4 b0
      x = fma(s_g[a] * s_g[q], mom(s_m, kM_b0, s_mul[a][q]), x);
    }
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (l == 0) s_c = x;
  }
  __syncthreads();
  // S' and h' of u' = [d; s x d]; (s x d)_a = s_a1 d_a2 - s_a2 d_a1
  if (tid < 36) {
    const int i = tid / 6, j = tid - i * 6;
    auto pk = [](int a, int b) { const int lo = min(a, b), hi = max(a, b); return lo == 0 ? hi : lo + hi + 1; };
    auto V = [&](int f, int a, int b) { return s_V[f * 6 + pk(a, b)]; };
    double x;
    if (i < 3 && j < 3) {
      x = V(0, i, j);
    } else if (i >= 3 && j >= 3) {
      const int a = i - 3, b = j - 3;
      const int a1 = (a + 1) % 3, a2 = (a + 2) % 3, b1 = (b + 1) % 3, b2 = (b + 2) % 3;
      x = (V(4 + pk(a1, b1), a2, b2) - V(4 + pk(a1, b2), a2, b1)) - (V(4 + pk(a2, b1), a1, b2) - V(4 + pk(a2, b2), a1, b1));
    } else {
      const int a = max(i, j) - 3, b = min(i, j), a1 = (a + 1) % 3, a2 = (a + 2) % 3;
      x = V(1 + a1, a2, b) - V(1 + a2, a1, b);
    }
    s_S[tid] = x;
  } else if (tid >= 64 && tid < 70) {
    const int i = tid - 64;
    if (i < 3) {
      s_h[i] = s_F[i];
    } else {
      const int a = i - 3, a1 = (a + 1) % 3, a2 = (a + 2) % 3;
      s_h[i] = s_F[(1 + a1) * 3 + a2] - s_F[(1 + a2) * 3 + a1];
    }
  } else if (tid >= 128 && tid < 200) {
    // N = M diag(R2, R2)
    const int which = (tid - 128) / 36, idx = (tid - 128) % 36, i = idx / 6, j = idx % 6;
    const double* M = which ? s_M2 : s_M1;
    const int b = j < 3 ? 0 : 3, c = j - b;
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) v = fma(M[i * 6 + b + k], T2[k * 4 + c], v);
    (which ? s_N2 : s_N1)[idx] = v;
  }
  __syncthreads();
  if (tid < 72) {
    const int which = tid / 36, idx = tid % 36, i = idx / 6, j = idx % 6;
    const double* M = which ? s_N2 : s_N1;
    double v = 0.0;
    for (int k = 0; k < 6; ++k) v += M[i * 6 + k] * s_S[k * 6 + j];
    (which ? s_T2 : s_T1)[idx] = v;
  }
  __syncthreads();
  double* out = contrib + (size_t)e * kBaContrib;
  if (tid < 108) {
    const int blk = tid / 36, idx = tid % 36, i = idx / 6, j = idx % 6;
    const double* Tm = (blk == 2) ? s_T2 : s_T1;
    const double* M = (blk == 0) ? s_N1 : s_N2;
    double v = 0.0;
    for (int k = 0; k < 6; ++k) v += Tm[i * 6 + k] * M[j * 6 + k];
    out[tid] = (blk == 1) ? -v : v;
  } else if (tid < 120) {
    const int which = (tid - 108) / 6, i = (tid - 108) % 6;
    const double* M = which ? s_N2 : s_N1;
    double v = 0.0;
    for (int k = 0; k < 6; ++k) v += M[i * 6 + k] * s_h[k];
    out[tid] = which ? -v : v;
  } else if (tid == 120) {
    out[120] = s_c;
  }
}

// Sum and maximum over the 64 lanes of a wave (butterfly; every lane gets the
// result, in a fixed order).
__device__ inline double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Flat element e < n (n + 1) / 2 of an n x n lower triangle, ordered by column
// descending: column k = n - 1 - m holds entries m (m + 1) / 2 ...
// m (m + 1) / 2 + m, rows k ... n - 1.
__device__ inline void triangle_index(int e, int n, int& i, int& k) {
  int m = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);
  while ((m + 1) * (m + 2) / 2 <= e) ++m;
  while (m * (m + 1) / 2 > e) --m;
  k = n - 1 - m;
  i = k + (e - m * (m + 1) / 2);
}

// Lane l's value of v (l uniform), moved through scalar registers.
__device__ __forceinline__ double readlane_f64(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum and maximum over the four waves of a solve block (waves in order);
// every thread calls them and gets the result.  The leading barrier keeps a
// previous call's readers ahead of this call's writers.
__device__ inline double block_sum4(double v, double* s_red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  return ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
}
__device__ inline double block_max4(double v, double* s_red) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmax(fmax(s_red[0], s_red[1]), fmax(s_red[2], s_red[3]));
}

// H, g and F at the poses Xe from the edge blocks: one wave per 6x6 block
// (fi, fj) of H, then one per 6-block of g (the first also sums F); every sum
// runs over the edges in index order.  H goes to the buffer that is not the
// current linearisation.  An edge adds one 6x6 (or 6) block of its contribution
// or nothing, so the wave first lists the edges that do, 64 at a time, then adds
// them with eight loads in flight (walking the edges one by one, each load behind
// the test of its edge, took 27 us at 66 edges, this 8.4).
__global__ __launch_bounds__(64) void ba_assemble_kernel(BaDev* __restrict__ ba, const BaEdge* __restrict__ edges,
                                                         const double* __restrict__ contrib,
                                                         double* __restrict__ Hbuf) {
  if (ba->done || !ba->eval_pending) return;
  const int nf = ba->nfree, n = ba->n, E = ba->n_edges;
  const int b = blockIdx.x, t = threadIdx.x;
  double* Hn = Hbuf + (size_t)(1 - ba->h_cur) * kBaMaxDof * kBaMaxDof;
  const bool hblock = b < nf * nf;
  const int fi = hblock ? b / nf : b - nf * nf;
  const int fj = hblock ? b - (b / nf) * nf : 0;
  const int a = t / 6, c = t % 6;
  __shared__ int s_at[kBaMaxEdges];    // offset of a listed edge's block, -1 - offset: transposed
  __shared__ int s_on[kBaMaxEdges];    // the edges that are on (F)
  int listed = 0, n_on = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + t;
    bool on = false, use = false;
    int at = 0;
    if (e < E) {
      const BaEdge& ed = edges[e];
      on = ed.on != 0;
      const int o1 = on ? ba->free_idx[ed.f1] : -2, o2 = on ? ba->free_idx[ed.f2] : -2;
      at = e * kBaContrib;
      if (hblock) {
        if (fi == fj) {
          use = o1 == fi || o2 == fi;
          if (o1 != fi) at += 72;
        } else {
          use = (o1 == fi && o2 == fj) || (o2 == fi && o1 == fj);
          at += 36;
          if (o1 != fi) at = -1 - at;
        }
      } else {
        use = o1 == fi || o2 == fi;
        at += o1 == fi ? 108 : 114;
      }
    }
    const uint64_t m = __ballot(use), mo = __ballot(on), below = (1ull << t) - 1ull;
    if (use) s_at[listed + __popcll(m & below)] = at;
    if (on) s_on[n_on + __popcll(mo & below)] = e * kBaContrib + 120;
    listed += __popcll(m);
    n_on += __popcll(mo);
  }
  __syncthreads();
  double s = 0.0;
  if (hblock ? t < 36 : t < 6) {
#pragma unroll 8
    for (int q = 0; q < listed; ++q) {
      const int at = s_at[q];
      s += hblock ? (at >= 0 ? contrib[at + a * 6 + c] : contrib[-1 - at + c * 6 + a]) : contrib[at + t];
    }
  } else if (!hblock && t == 6 && fi == 0) {
#pragma unroll 8
    for (int q = 0; q < n_on; ++q) s += 0.5 * contrib[s_on[q]];
  }
  if (hblock) {
    if (t < 36) Hn[(size_t)(6 * fi + a) * n + 6 * fj + c] = s;
  } else if (t < 6) {
    ba->gn[6 * fi + t] = s;
  } else if (t == 6 && fi == 0) {
    ba->Fn = s;
  }
}

// One block of four waves: the Levenberg-Marquardt decision on an evaluated
// candidate, then the next candidate (or the end of the solve).  Scalars of
// the schedule are kept uniform in every thread (block-wide reductions) and
// written back by thread 0; thread i < n holds entry i of the gradient; the
// damped system is factored in LDS (right-looking Cholesky, the trailing
// update over all four waves), the triangular solves run in wave 0 with the
// right-hand side in registers (rows lane and lane + 64).
__global__ __launch_bounds__(kSolveThreads) void ba_solve_kernel(BaDev* __restrict__ ba, double* __restrict__ Hbuf) {
  if (ba->done || !ba->eval_pending) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = ba->n;
  const int ld = n | 1;  // odd row stride in LDS
  __shared__ double s_A[kBaMaxDof * (kBaMaxDof + 1)];
  __shared__ double s_d[kBaMaxDof];
  __shared__ double s_g[kBaMaxDof];
  __shared__ double s_inv[kBaMaxDof];  // 1 / L(j, j)
  __shared__ double s_red[kSolveThreads / 64];
  __shared__ int s_fail;
  const bool candidate = ba->eval_is_candidate != 0;
  int cur = ba->h_cur;
  double mu = ba->mu, v = ba->v, F = ba->F;
  const double Fn = ba->Fn;
  int lm_iter = ba->lm_iter, lm_stop = ba->lm_stop;
  int accepted_total = ba->accepted_total, evals_total = ba->evals_total;
  const int max_lm = ba->iters_per_solve;
  bool take = !candidate;
  if (candidate) {
    // predicted decrease -(g.d + d.H.d / 2) at the current linearisation,
    // H read once, coalesced
    const double* H = Hbuf + (size_t)cur * kBaMaxDof * kBaMaxDof;
    if (tid < n) s_d[tid] = ba->d[tid];
    __syncthreads();
    double part = 0.0;
    // eight loads in flight per thread
#pragma unroll 8
    for (int idx = tid; idx < n * n; idx += kSolveThreads) {
      const int i = idx / n, j = idx - i * n;
      part += s_d[i] * H[idx] * s_d[j];
    }
    part *= 0.5;
    if (tid < n) part += s_d[tid] * ba->g[tid];
    const double pred = -block_sum4(part, s_red);
    const double rho = pred > 0.0 ? (F - Fn) / pred : -1.0;
    evals_total++;
    if (rho > 1e-3) {
      const double rel = fabs(F - Fn) / fmax(F, 1e-300);
      mu = fmin(mu / fmax(1.0 / 3.0, 1.0 - pow(2.0 * rho - 1.0, 3.0)), 1e16);
      v = 2.0;
      accepted_total++;
      if (rel < 1e-5) lm_stop = 1;
      take = true;
    } else {
      mu /= v;
      v *= 2.0;
    }
    lm_iter++;
  }
  // current linearisation: thread i's gradient entry, poses X
  const double* Xs = (take && candidate) ? ba->Xe : ba->X;
  double g = 0.0;
  if (take) {
    if (tid < n) {
      g = ba->gn[tid];
      ba->g[tid] = g;
    }
    F = Fn;
    cur = 1 - cur;
  } else {
    if (tid < n) g = ba->g[tid];
  }
  if (tid < n) s_g[tid] = g;
  double xs2 = 0.0;
  for (int i = tid; i < ba->n_frames * 12; i += kSolveThreads) {
    const double x = Xs[i];
    xs2 += x * x;
    if (take && candidate) ba->X[i] = x;
  }
  const double xn = sqrt(block_sum4(xs2, s_red));
  const double* H = Hbuf + (size_t)cur * kBaMaxDof * kBaMaxDof;
  int pending = 0;
  // every thread holds the same control values (block-wide reductions), so
  // the loop and its barriers are uniform
  while (true) {
    if (lm_stop || lm_iter >= max_lm) break;
    const double gmax = block_max4(fabs(g), s_red);
    if (gmax < 1e-5) {
      lm_stop = 1;
      break;
    }
#pragma unroll 8
    for (int idx = tid; idx < n * n; idx += kSolveThreads) {
      const int i = idx / n, j = idx - i * n;
      double x = H[idx];
      if (i == j) x += fmin(fmax(x, 1e-6), 1e32) / mu;
      s_A[i * ld + j] = x;
    }
    __syncthreads();
    // blocked right-looking Cholesky, kChol columns a block: wave 0 factors
    // the block's panel (rows from the block on, its columns) in registers,
    // rows j0 + lane and j0 + lane + 64 a lane, entries of the block's own rows
    // by readlane; then all four waves subtract the block's columns from the
    // trailing triangle in 2x2 tiles, per element in the same order as column
    // by column (the result is the unblocked one bit for bit).  What is left
    // above the diagonal is not read.  The diagonal's reciprocal goes to s_inv
    bool fail = false;
    for (int j0 = 0; j0 < n; j0 += kChol) {
      const int jb = min(kChol, n - j0);
      if (wave == 0) {
        const int r0 = j0 + lane, r1 = r0 + 64;
        double* R0 = s_A + min(r0, n - 1) * ld;
        double* R1 = s_A + min(r1, n - 1) * ld;
        double p0[kChol], p1[kChol];
#pragma unroll
        for (int c = 0; c < kChol; ++c) {
          const int j = min(j0 + c, n - 1);
          p0[c] = R0[j];
          p1[c] = R1[j];
        }
        int f = 0;
#pragma unroll
        for (int c = 0; c < kChol; ++c) {
          if (c >= jb || f) break;  // uniform
          const double ajj = readlane_f64(p0[c], c);
          if (!(ajj > 0.0)) {
            f = 1;
            break;
          }
          const double inv = 1.0 / sqrt(ajj);
          if (lane == 0) s_inv[j0 + c] = inv;
          if (lane > c) p0[c] *= inv;
          p1[c] *= inv;
#pragma unroll
          for (int k = c + 1; k < kChol; ++k) {
            const double lkj = readlane_f64(p0[c], k);
            p0[k] -= p0[c] * lkj;
            p1[k] -= p1[c] * lkj;
          }
        }
#pragma unroll
        for (int c = 0; c < kChol; ++c) {
          if (c >= jb) break;
          if (r0 < n) R0[j0 + c] = p0[c];
          if (r1 < n) R1[j0 + c] = p1[c];
        }
        if (lane == 0) s_fail = f;
      }
      __syncthreads();
      if (s_fail) {  // uniform
        fail = true;
        break;
      }
      // 2x2 tiles, those on and below the diagonal in flat order; n and the
      // block are even, and where columns are left the block is a whole one.
      // Single elements, four a thread with an index each, and the panel through
      // LDS: 77 us a launch at 66 dof, so 50
      const int base = j0 + jb, T = (n - base) / 2;
      for (int e = tid; e < T * (T + 1) / 2; e += kSolveThreads) {
        int i, k;
        triangle_index(e, T, i, k);
        i = base + 2 * i;
        k = base + 2 * k;
        double* Ai = s_A + i * ld;
        double* Bi = Ai + ld;
        const double* Ak = s_A + k * ld + j0;
        const double* Bk = Ak + ld;
        double x00 = Ai[k], x01 = Ai[k + 1], x10 = Bi[k], x11 = Bi[k + 1];
#pragma unroll
        for (int c = 0; c < kChol; ++c) {
          const double a0 = Ai[j0 + c], a1 = Bi[j0 + c], b0 = Ak[c], b1 = Bk[c];
          x00 -= a0 * b0;
          x01 -= a0 * b1;
          x10 -= a1 * b0;
          x11 -= a1 * b1;
        }
        Ai[k] = x00;
        Ai[k + 1] = x01;
        Bi[k] = x10;
        Bi[k + 1] = x11;
      }
      __syncthreads();
    }
    if (fail) {
      mu /= v;
      v *= 2.0;
      lm_iter++;
      __syncthreads();
      continue;
    }
    // L y = -g, then L^T d = y: one wave, rows r and r + 64 per lane; the
    // solved entry moves by readlane, and the L entries and reciprocals of
    // kTri steps are read from LDS ahead of the steps that use them (rows
    // clamped to n - 1 for the loads; those values are not used)
    if (wave == 0) {
      const int r0 = lane, r1 = lane + 64;
      const int c0 = min(r0, n - 1), c1 = min(r1, n - 1);
      double b0 = r0 < n ? -s_g[r0] : 0.0, b1 = r1 < n ? -s_g[r1] : 0.0;
      for (int i0 = 0; i0 < n; i0 += kTri) {
        double l0[kTri], l1[kTri], sv[kTri];
#pragma unroll
        for (int u = 0; u < kTri; ++u) {
          const int i = min(i0 + u, n - 1);
          l0[u] = s_A[c0 * ld + i];
          l1[u] = s_A[c1 * ld + i];
          sv[u] = s_inv[i];
        }
#pragma unroll
        for (int u = 0; u < kTri; ++u) {
          const int i = i0 + u;
          if (i >= n) break;  // uniform
          const double bi = i < 64 ? readlane_f64(b0, i) : readlane_f64(b1, i - 64);
          const double yi = bi * sv[u];
          if (r0 == i) b0 = yi;
          if (r1 == i) b1 = yi;
          if (r0 > i && r0 < n) b0 -= l0[u] * yi;
          if (r1 > i && r1 < n) b1 -= l1[u] * yi;
        }
      }
      for (int i0 = n - 1; i0 >= 0; i0 -= kTri) {
        double l0[kTri], l1[kTri], sv[kTri];
#pragma unroll
        for (int u = 0; u < kTri; ++u) {
          const int i = max(i0 - u, 0);
          l0[u] = s_A[i * ld + c0];
          l1[u] = s_A[i * ld + c1];
          sv[u] = s_inv[i];
        }
#pragma unroll
        for (int u = 0; u < kTri; ++u) {
          const int i = i0 - u;
          if (i < 0) break;  // uniform
          const double bi = i < 64 ? readlane_f64(b0, i) : readlane_f64(b1, i - 64);
          const double xi = bi * sv[u];
          if (r0 == i) b0 = xi;
          if (r1 == i) b1 = xi;
          if (r0 < i) b0 -= l0[u] * xi;
          if (r1 < i) b1 -= l1[u] * xi;
        }
      }
      if (r0 < n) s_d[r0] = b0;
      if (r1 < n) s_d[r1] = b1;
    }
    __syncthreads();
    const double dd = tid < n ? s_d[tid] * s_d[tid] : 0.0;
    const double dn = sqrt(block_sum4(dd, s_red));
    if (dn < 1e-5 * (xn + 1e-5)) {
      lm_stop = 1;
      break;
    }
    if (tid < n) ba->d[tid] = s_d[tid];
    for (int f = tid; f < ba->n_frames; f += kSolveThreads) {
      const int o = ba->free_idx[f];
      if (o >= 0) pose_plus(Xs + 12 * f, s_d + 6 * o, ba->Xe + 12 * f);
      else
        for (int i = 0; i < 12; ++i) ba->Xe[12 * f + i] = Xs[12 * f + i];
    }
    pending = 1;
    break;
  }
  if (tid == 0) {
    ba->h_cur = cur;
    ba->mu = mu;
    ba->v = v;
    ba->F = F;
    ba->lm_iter = lm_iter;
    ba->lm_stop = lm_stop;
    ba->accepted_total = accepted_total;
    ba->evals_total = evals_total;
    ba->eval_pending = pending;
    ba->eval_is_candidate = pending;
  }
}

// Per-edge lengthscale (BinaryStateGPU::update_ell, IRLS_State_GPU.cpp:
// 117-146, mode 0), pose change (IRLS.cpp:99-108) and convergence
// (IRLS.cpp:325-339).  One wave: lanes over edges and frames.
__global__ __launch_bounds__(64) void ba_finish_kernel(BaDev* __restrict__ ba, BaEdge* __restrict__ edges) {
  if (ba->done) return;
  const int lane = threadIdx.x;
  int not_min = 0;
  for (int e = lane; e < ba->n_edges; e += 64) {
    BaEdge& ed = edges[e];
    ed.iters_per_ell++;
    if (ed.nnz_last > 0 && ed.nnz <= ed.nnz_last && ed.iters_per_ell / ba->iter_per_ell > 0) {
      ed.ell = ed.ell * (double)ba->decay_f;
      ed.iters_per_ell = 0;
    }
    if (ed.ell < ba->ell_min) ed.ell = ba->ell_min;
    else if (ed.ell > ba->ell_max) ed.ell = ba->ell_max;
    if (!(fabsf((float)ed.ell - ba->ell_min_f) < 1e-4f)) not_min = 1;
  }
  double change = 0.0;
  for (int f = lane; f < ba->n_frames; f += 64) {
    const double* A = ba->Xold + 12 * f;
    const double* B = ba->X + 12 * f;
    double R[9], t[3];
    for (int r = 0; r < 3; ++r) {
      for (int c = 0; c < 3; ++c)
        R[r * 3 + c] = A[0 * 4 + r] * B[0 * 4 + c] + A[1 * 4 + r] * B[1 * 4 + c] + A[2 * 4 + r] * B[2 * 4 + c];
      t[r] = A[0 * 4 + r] * (B[3] - A[3]) + A[1 * 4 + r] * (B[7] - A[7]) + A[2 * 4 + r] * (B[11] - A[11]);
    }
    change += se3_log_norm(R, t);
  }
  change = wave_sum(change);
  const bool all_min = wave_max((double)not_min) == 0.0;
  if (lane == 0) {
    ba->change = change;
    ba->iter++;
    if ((all_min && change < 1e-5) || ba->iter >= ba->max_iters) ba->done = 1;
  }
}

// ---------------------------------------------------------------------------
// Host
// ---------------------------------------------------------------------------

template <class T>
static T* as(DevBuf& b) {
  return reinterpret_cast<T*>(b.p);
}

enum {
  BA_PAIRS = 0, BA_COUNTS, BA_OVF, BA_STATE, BA_PROBS, BA_PART_A, BA_PART_OVF, BA_PART_CNT,
  BA_DEV, BA_EDGES, BA_H, BA_HN, BA_MOM_PART, BA_CONTRIB, BA_PAIR_IDS
};

// Six buffers per frame: sorted source (pos, feat, sem, geo), grid store and
// grid header.
constexpr int kFrameBufs = 6;

static cvo_status validate_frames(cvo_ctx* ctx, int n_frames, const cvo_dcloud* const* frames, const double* poses,
                                  const uint8_t* hold_const, int n_edges, const int32_t* edges, int* nfree_out) {
  const cvo_params& p = ctx->params;
  if (n_frames <= 0 || !frames || !poses) return set_err(ctx, CVO_ERR_INVALID_ARG, "no frames");
  if (n_frames > kBaMaxFrames) return set_err(ctx, CVO_ERR_LIMIT, "at most 64 frames");
  if (n_edges < 0 || n_edges > kBaMaxEdges) return set_err(ctx, CVO_ERR_LIMIT, "edge count out of [0, 4096]");
  if (n_edges > 0 && !edges) return set_err(ctx, CVO_ERR_INVALID_ARG, "null edge list");
  for (int f = 0; f < n_frames; ++f) {
    if (!frames[f]) return set_err(ctx, CVO_ERR_INVALID_ARG, "null frame");
    if (frames[f]->n == 0) return set_err(ctx, CVO_ERR_EMPTY, "empty frame");
    if (frames[f]->F != frames[0]->F || frames[f]->K != frames[0]->K)
      return set_err(ctx, CVO_ERR_INVALID_ARG, "frames differ in feature or class dimension");
    for (int i = 0; i < 12; ++i)
      if (!std::isfinite(poses[12 * f + i])) return set_err(ctx, CVO_ERR_INVALID_ARG, "non-finite pose");
  }
  int nfree = 0;
  for (int f = 0; f < n_frames; ++f)
    if (!hold_const || !hold_const[f]) nfree++;
  if (nfree > kBaMaxFree) return set_err(ctx, CVO_ERR_LIMIT, "at most 20 frames may be free");
  for (int e = 0; e < n_edges; ++e) {
    const int a = edges[2 * e], b = edges[2 * e + 1];
    if (a < 0 || a >= n_frames || b < 0 || b >= n_frames || a == b)
      return set_err(ctx, CVO_ERR_INVALID_ARG, "edge frame index out of range or self edge");
    CVO_TRY(validate_pair(ctx, frames[a], frames[b]));
  }
  if (p.multiframe_num_neighbors < 1 || p.multiframe_num_neighbors > 1024)
    return set_err(ctx, CVO_ERR_LIMIT, "multiframe_num_neighbors must be in [1, 1024]");
  // the K-nearest search keeps at most KDTREE_K_SIZE per row (cukdtree.h:12,40)
  if (p.is_using_kdtree && p.multiframe_num_neighbors > kKnnMaxK)
    return set_err(ctx, CVO_ERR_LIMIT, "is_using_kdtree needs multiframe_num_neighbors <= 512");
  if (p.multiframe_iter_per_ell <= 0) return set_err(ctx, CVO_ERR_INVALID_ARG, "multiframe_iter_per_ell must be > 0");
  if (!(p.multiframe_ell_init > 0.0f) || !(p.multiframe_ell_min > 0.0f))
    return set_err(ctx, CVO_ERR_INVALID_ARG, "multiframe lengthscales must be positive");
  *nfree_out = nfree;
  return CVO_OK;
}


struct BaLaunch {
  BaDev* ba;
  BaEdge* edges;
  AssocProblem* probs;
  int n_edges, total_blocks, mom_rows, max_mom_blocks, lm_rounds, n_asm_blocks;
  double* part;     // blocks' moments; the edges' own where each edge has one block
  double* moments;
  double* contrib;
  double* H;  // two n x n halves: current linearisation and evaluation
  KConsts kc;
};

static void ba_assoc_phase(const BaLaunch& L, hipStream_t s) {
  hipLaunchKernelGGL(ba_prepare_kernel, dim3(1), dim3(256), 0, s, L.ba, L.edges, L.probs);
  if (L.n_edges > 0) {
    launch_assoc(L.probs, L.n_edges, L.total_blocks, L.kc, s);
    launch_overflow(L.probs, L.n_edges, L.kc, s);
  }
  hipLaunchKernelGGL(ba_edges_kernel, dim3(1), dim3(256), 0, s, L.ba, L.edges, L.probs);
}

// e0 / e1 (optional): events at the moment kernel's own start and end.
static void ba_moments_phase(const BaLaunch& L, hipStream_t s, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr) {
  const dim3 g(L.max_mom_blocks, L.n_edges), b(256);
  if (e0) hipExtLaunchKernelGGL(ba_moments_kernel, g, b, 0, s, e0, e1, 0, L.ba, L.edges, L.probs, L.part, L.mom_rows);
  else hipLaunchKernelGGL(ba_moments_kernel, g, b, 0, s, L.ba, L.edges, L.probs, L.part, L.mom_rows);
  if (L.part != L.moments)
    hipLaunchKernelGGL(ba_moments_sum_kernel, dim3(L.n_edges, (kMomUsed + 255) / 256), dim3(256), 0, s, L.ba, L.edges,
                       L.part, L.moments);
}

static void ba_lm_round(const BaLaunch& L, hipStream_t s) {
  hipLaunchKernelGGL(ba_eval_kernel, dim3(L.n_edges), dim3(384), 0, s, L.ba, L.edges, L.moments, L.contrib);
  hipLaunchKernelGGL(ba_assemble_kernel, dim3(L.n_asm_blocks), dim3(64), 0, s, L.ba, L.edges, L.contrib, L.H);
  hipLaunchKernelGGL(ba_solve_kernel, dim3(1), dim3(kSolveThreads), 0, s, L.ba, L.H);
}

static void ba_iteration(const BaLaunch& L, hipStream_t s) {
  ba_assoc_phase(L, s);
  if (L.n_edges > 0) {
    ba_moments_phase(L, s);
    for (int k = 0; k < L.lm_rounds; ++k) ba_lm_round(L, s);
  }
  hipLaunchKernelGGL(ba_finish_kernel, dim3(1), dim3(64), 0, s, L.ba, L.edges);
}

}  // namespace cvo

using namespace cvo;

// Under a workspace limit the moment partials are given back at the end: other
// calls may need the room that this one used.
struct PartHolder {
  cvo_ctx* ctx;
  DevBuf& b;
  void release() {
    if (ctx->ws_limit > 0) free_buf(ctx, b);
  }
  ~PartHolder() { release(); }
};

extern "C" cvo_status cvo_align_multiframe(cvo_ctx* ctx, int32_t n_frames, const cvo_dcloud* const* frames,
                                           double* poses, const uint8_t* hold_const, int32_t n_edges,
                                           const int32_t* edges, cvo_assoc* per_edge, double* seconds,
                                           int32_t* iters, double* per_iter_seconds, int32_t max_iter_records) {
  if (!ctx) return CVO_ERR_INVALID_ARG;
  ActiveCall busy(ctx);
  if (per_edge)
    for (int e = 0; e < n_edges; ++e) std::memset(&per_edge[e], 0, sizeof(cvo_assoc));
  if (seconds) *seconds = 0.0;
  if (iters) *iters = 0;
  int nfree = 0;
  CVO_TRY(validate_frames(ctx, n_frames, frames, poses, hold_const, n_edges, edges, &nfree));
  const cvo_params& p = ctx->params;
  hipStream_t st = ctx->stream;
  const auto t_start = std::chrono::steady_clock::now();
  KConsts kc = make_kconsts(p, frames[0]->F, frames[0]->K, MODE_BA);
  int64_t all_rows = 1;
  for (int e = 0; e < n_edges; ++e) all_rows += frames[edges[2 * e]]->n;
  apply_tuning(ctx, kc, all_rows);  // one batched launch over the edges
  const int rb = rows_per_block(kc.max_group);

  // frames that are sources / targets of some edge
  std::vector<char> is_src(n_frames, 0), is_tgt(n_frames, 0);
  for (int e = 0; e < n_edges; ++e) {
    is_src[edges[2 * e]] = 1;
    is_tgt[edges[2 * e + 1]] = 1;
  }
  float max_world = 0.0f, max_t = 0.0f;
  for (int f = 0; f < n_frames; ++f) {
    const double* T = poses + 12 * f;
    const float tn = (float)std::sqrt(T[3] * T[3] + T[7] * T[7] + T[11] * T[11]);
    max_world = std::max(max_world, frames[f]->max_norm + tn);
    max_t = std::max(max_t, tn);
  }
  if (ctx->b_frames.size() < (size_t)kFrameBufs * n_frames) ctx->b_frames.resize((size_t)kFrameBufs * n_frames);
  std::vector<GridHost> grids(n_frames);
  const float ell_hi = std::max(p.multiframe_ell_init * 1.2f, p.multiframe_ell_min);
  const float ell_lo = std::min(p.multiframe_ell_min, p.multiframe_ell_init);
  const std::vector<float> hs = level_sizes(kc, ell_hi, ell_lo, max_world * 1.05f, max_t * 1.05f + 1.0f, kc.min_scale);
  for (int f = 0; f < n_frames; ++f) {
    DevBuf* fb = &ctx->b_frames[(size_t)kFrameBufs * f];
    if (is_src[f]) CVO_TRY(prepare_source_into(ctx, frames[f], fb[0], fb[1], fb[2], fb[3]));
    if (is_tgt[f]) CVO_TRY(build_grid_into(ctx, frames[f], hs, grids[f], fb[4], fb[5]));
  }

  // per-edge association problems
  const int cap = p.multiframe_num_neighbors;
  size_t tot_rows = 0;
  int total_blocks = 0, max_rows = 1;
  std::vector<size_t> row_off(n_edges + 1, 0);
  for (int e = 0; e < n_edges; ++e) {
    const int n = frames[edges[2 * e]]->n;
    row_off[e + 1] = row_off[e] + (size_t)n;
    total_blocks += (n + rb - 1) / rb;
    max_rows = std::max(max_rows, n);
  }
  tot_rows = row_off[n_edges];
  const size_t E1 = (size_t)std::max(n_edges, 1);
  DevBuf* B = ctx->b_ba;
  CVO_TRY(ensure(ctx, B[BA_PAIRS], sizeof(float4) * std::max<size_t>(tot_rows, 1) * cap));
  CVO_TRY(ensure(ctx, B[BA_COUNTS], sizeof(uint32_t) * std::max<size_t>(tot_rows, 1)));
  CVO_TRY(ensure(ctx, B[BA_OVF], sizeof(uint32_t) * std::max<size_t>(tot_rows, 1)));
  CVO_TRY(ensure(ctx, B[BA_STATE], sizeof(ProblemState) * E1));
  CVO_TRY(ensure(ctx, B[BA_PROBS], sizeof(AssocProblem) * E1));
  CVO_TRY(ensure(ctx, B[BA_PART_A], sizeof(double) * 8 * (size_t)std::max(total_blocks, 1)));
  CVO_TRY(ensure(ctx, B[BA_PART_OVF], sizeof(double) * 10 * kOvfBlocks * E1));
  CVO_TRY(ensure(ctx, B[BA_PART_CNT], sizeof(uint32_t) * 2 * (size_t)std::max(total_blocks, 1)));
  CVO_TRY(ensure(ctx, B[BA_DEV], sizeof(BaDev)));
  CVO_TRY(ensure(ctx, B[BA_EDGES], sizeof(BaEdge) * E1));
  CVO_TRY(ensure(ctx, B[BA_H], sizeof(double) * 2 * kBaMaxDof * kBaMaxDof));
  CVO_TRY(ensure(ctx, B[BA_CONTRIB], sizeof(double) * kBaContrib * E1));
  // the export needs each stored pair's target (its sorted position)
  if (per_edge) CVO_TRY(ensure(ctx, B[BA_PAIR_IDS], sizeof(uint32_t) * std::max<size_t>(tot_rows, 1) * cap));
  // Moment blocks of kMomRows rows; of twice as many, and so on, where a workspace
  // limit would not hold their partials.  One block an edge needs none: it writes
  // the edge's moments, in memory that the association has anyway.
  int mom_rows = kMomRows;
  auto mom_blocks = [&](int n) { return (n + mom_rows - 1) / mom_rows; };
  auto part_bytes = [&]() {
    size_t blocks = 0;
    if (max_rows > mom_rows)
      for (int e = 0; e < n_edges; ++e) blocks += (size_t)mom_blocks(frames[edges[2 * e]]->n);
    return sizeof(double) * kMomUsed * blocks;
  };
  if (ctx->ws_limit > 0) {
    const size_t held = ctx->ws_bytes - B[BA_MOM_PART].cap;
    const size_t room = ctx->ws_limit > held ? (ctx->ws_limit - held) / 5 * 4 : 0;  // the arena's headroom
    while (part_bytes() > room) mom_rows *= 2;
  }
  PartHolder part_holder{ctx, B[BA_MOM_PART]};
  if (part_bytes() > 0) CVO_TRY(ensure(ctx, B[BA_MOM_PART], part_bytes()));
  CVO_HIP(ctx, hipMemsetAsync(B[BA_OVF].p, 0, sizeof(uint32_t) * std::max<size_t>(tot_rows, 1), st));
  CVO_HIP(ctx, hipMemsetAsync(B[BA_STATE].p, 0, sizeof(ProblemState) * E1, st));

  std::vector<AssocProblem> hp(E1);
  std::vector<BaEdge> he(E1);
  int blk = 0, mom_blk = 0;
  for (int e = 0; e < n_edges; ++e) {
    const int f1 = edges[2 * e], f2 = edges[2 * e + 1];
    const cvo_dcloud* s = frames[f1];
    const cvo_dcloud* t = frames[f2];
    DevBuf* sb = &ctx->b_frames[(size_t)kFrameBufs * f1];
    const int n = s->n;
    const int nb = (n + rb - 1) / rb;
    AssocProblem& P = hp[e];
    std::memset(&P, 0, sizeof(P));
    P.src_pos = as<float4>(sb[0]);
    P.src_feat = s->feat ? as<float>(sb[1]) : nullptr;
    P.src_sem = s->sem ? as<float>(sb[2]) : nullptr;
    P.src_geo = s->geo ? as<float>(sb[3]) : nullptr;
    P.n_src = n;
    P.n_tgt = t->n;
    P.grid = grids[f2].dev_ptr;
    P.tgt_xyz = t->xyz;
    P.tgt_feat = t->feat;
    P.tgt_sem = t->sem;
    P.tgt_geo = t->geo;
    P.st = as<ProblemState>(B[BA_STATE]) + e;
    P.pairs = nullptr;
    P.pairs4 = as<float4>(B[BA_PAIRS]) + row_off[e] * cap;
    P.pair_ids = per_edge ? as<uint32_t>(B[BA_PAIR_IDS]) + row_off[e] * cap : nullptr;
    P.counts = as<uint32_t>(B[BA_COUNTS]) + row_off[e];
    P.ovf_stamp = as<uint32_t>(B[BA_OVF]) + row_off[e];
    P.cap_alloc = cap;
    P.block_begin = blk;
    P.n_blocks = nb;
    P.part_a = as<double>(B[BA_PART_A]) + (size_t)blk * 8;
    P.part_ovf = as<double>(B[BA_PART_OVF]) + (size_t)e * kOvfBlocks * 10;
    P.part_s = nullptr;
    P.part_cnt = as<uint32_t>(B[BA_PART_CNT]) + (size_t)blk * 2;
    blk += nb;
    BaEdge& ed = he[e];
    std::memset(&ed, 0, sizeof(ed));
    ed.ell = (double)p.multiframe_ell_init;
    ed.f1 = f1;
    ed.f2 = f2;
    ed.K = cap;
    ed.n_rows = n;
    ed.n_blocks = mom_blocks(n);
    ed.part0 = mom_blk;
    mom_blk += ed.n_blocks;
  }
  if (n_edges > 0) {
    CVO_HIP(ctx, hipMemcpyAsync(B[BA_PROBS].p, hp.data(), sizeof(AssocProblem) * n_edges, hipMemcpyHostToDevice, st));
    CVO_HIP(ctx, hipMemcpyAsync(B[BA_EDGES].p, he.data(), sizeof(BaEdge) * n_edges, hipMemcpyHostToDevice, st));
  }
  BaDev* hb = new BaDev;
  std::memset(hb, 0, sizeof(BaDev));
  hb->n_frames = n_frames;
  hb->n_edges = n_edges;
  hb->nfree = nfree;
  hb->n = 6 * nfree;
  hb->max_iters = p.multiframe_max_iters;
  hb->iters_per_solve = p.multiframe_iterations_per_solve;
  hb->K_init = cap;
  hb->min_nonzeros = p.multiframe_min_nonzeros;
  hb->iter_per_ell = p.multiframe_iter_per_ell;
  hb->ell_min_f = p.multiframe_ell_min;
  hb->decay_f = p.multiframe_ell_decay_rate;
  hb->rq_coef = kc.rq_coef;
  hb->pol = kc.pol;
  hb->ell_min = (double)p.multiframe_ell_min;
  hb->ell_max = (double)p.multiframe_ell_init * 1.2;
  int o = 0;
  for (int f = 0; f < n_frames; ++f) {
    hb->free_idx[f] = (!hold_const || !hold_const[f]) ? o++ : -1;
    if (hb->free_idx[f] >= 0) hb->frame_of_free[hb->free_idx[f]] = f;
    hb->frame_norm[f] = frames[f]->max_norm;
    for (int i = 0; i < 12; ++i) hb->X[12 * f + i] = poses[12 * f + i];
  }
  hb->done = p.multiframe_max_iters <= 0 ? 1 : 0;
  hipError_t ce = hipMemcpyAsync(B[BA_DEV].p, hb, sizeof(BaDev), hipMemcpyHostToDevice, st);
  hipError_t se = hipStreamSynchronize(st);  // hb is pageable host memory
  delete hb;
  if (ce != hipSuccess) return hip_check(ctx, ce, "BA state upload");
  if (se != hipSuccess) return hip_check(ctx, se, "BA state upload");

  BaLaunch L;
  L.ba = as<BaDev>(B[BA_DEV]);
  L.edges = as<BaEdge>(B[BA_EDGES]);
  L.probs = as<AssocProblem>(B[BA_PROBS]);
  L.n_edges = n_edges;
  L.total_blocks = total_blocks;
  L.mom_rows = mom_rows;
  L.max_mom_blocks = mom_blocks(max_rows);
  L.lm_rounds = std::max(0, p.multiframe_iterations_per_solve) + 1;
  L.n_asm_blocks = std::max(1, nfree * nfree + nfree);
  L.moments = as<double>(B[BA_PART_OVF]);
  L.part = part_bytes() > 0 ? as<double>(B[BA_MOM_PART]) : L.moments;
  L.contrib = as<double>(B[BA_CONTRIB]);
  L.H = as<double>(B[BA_H]);
  L.kc = kc;

  CVO_TRY(pinned(ctx, 64));
  volatile int32_t* flag = reinterpret_cast<volatile int32_t*>(ctx->pinned);
  const char* ng = std::getenv("CVO_NO_GRAPH");
  const bool use_graph = !(ng && ng[0] && ng[0] != '0') && !ctx->profiling;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  if (use_graph) {
    CVO_HIP(ctx, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    ba_iteration(L, st);
    hipError_t e1 = hipStreamEndCapture(st, &graph);
    if (e1 != hipSuccess) return hip_check(ctx, e1, "hipStreamEndCapture");
    hipError_t e2 = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (e2 != hipSuccess) {
      (void)hipGraphDestroy(graph);
      return hip_check(ctx, e2, "hipGraphInstantiate");
    }
  }
  CVO_TRY(ensure_events(ctx, 24));
  hipEvent_t ev[6];
  for (int i = 0; i < 6; ++i) ev[i] = ctx->ev_pool[16 + i];
  cvo_status status = CVO_OK;
  const int max_outer = std::max(0, p.multiframe_max_iters) + 1;
  for (int it = 0; it < max_outer; ++it) {
    const auto ti0 = std::chrono::steady_clock::now();
    hipError_t le = hipSuccess;
    if (use_graph) {
      le = hipGraphLaunch(exec, st);
    } else if (ctx->profiling) {
      (void)hipEventRecord(ev[0], st);
      hipLaunchKernelGGL(ba_prepare_kernel, dim3(1), dim3(256), 0, st, L.ba, L.edges, L.probs);
      // association kernel timed alone (events at its own start and end)
      if (n_edges > 0) launch_assoc(L.probs, n_edges, total_blocks, kc, st, nullptr, ev[1], ev[2]);
      else (void)hipEventRecord(ev[1], st), (void)hipEventRecord(ev[2], st);
      if (n_edges > 0) {
        launch_overflow(L.probs, n_edges, kc, st);
      }
      hipLaunchKernelGGL(ba_edges_kernel, dim3(1), dim3(256), 0, st, L.ba, L.edges, L.probs);
      (void)hipEventRecord(ev[3], st);
      // algorithmic bytes: association reads both clouds' points and writes
      // the pairs; a pair pass reads the stored pairs, the target positions
      // they name and the source rows
      std::vector<BaEdge> eh(n_edges);
      if (n_edges > 0)
        (void)hipMemcpyAsync(eh.data(), L.edges, sizeof(BaEdge) * n_edges, hipMemcpyDeviceToHost, st);
      (void)hipStreamSynchronize(st);
      float m_assoc = 0, m_ovf = 0;
      (void)hipEventElapsedTime(&m_assoc, ev[1], ev[2]);
      (void)hipEventElapsedTime(&m_ovf, ev[2], ev[3]);
      double pair_bytes = 0.0;
      const double per_pt = 12.0 + (kc.use_col ? 4.0 * kc.F : 0.0) + (kc.use_sem ? 4.0 * kc.Ks : 0.0);
      for (int e = 0; e < n_edges; ++e) {
        const double S = (double)eh[e].nnz;
        ctx->stats.bytes[CVO_KSTAT_ASSOC] += per_pt * (frames[eh[e].f1]->n + frames[eh[e].f2]->n) + 16.0 * S +
                                             4.0 * frames[eh[e].f1]->n;
        ctx->stats.pairs_stored += S;
        if (eh[e].on) pair_bytes += 16.0 * S + 20.0 * eh[e].n_rows;
      }
      float ms_pair = 0.0f, ms_solve = 0.0f;
      int pair_launches = 0, solve_launches = 0;
      auto pending = [&]() {
        int32_t pend = 0;
        (void)hipMemcpyAsync(&pend, &L.ba->eval_pending, sizeof(int32_t), hipMemcpyDeviceToHost, st);
        (void)hipStreamSynchronize(st);
        return pend != 0;
      };
      if (n_edges > 0) {
        // the moment kernel timed alone
        const bool work = pending();
        ba_moments_phase(L, st, ev[4], ev[5]);
        (void)hipStreamSynchronize(st);
        if (work) {
          (void)hipEventElapsedTime(&ms_pair, ev[4], ev[5]);
          pair_launches = 1;
          ctx->stats.bytes[CVO_KSTAT_BA_PAIR] += pair_bytes;
        }
      }
      for (int k = 0; k < (n_edges > 0 ? L.lm_rounds : 0); ++k) {
        const bool work = pending();
        (void)hipEventRecord(ev[4], st);
        ba_lm_round(L, st);
        (void)hipEventRecord(ev[3], st);
        (void)hipEventSynchronize(ev[3]);
        float b = 0;
        (void)hipEventElapsedTime(&b, ev[4], ev[3]);
        if (work) {
          ms_solve += b;
          solve_launches++;
        }
      }
      hipLaunchKernelGGL(ba_finish_kernel, dim3(1), dim3(64), 0, st, L.ba, L.edges);
      ctx->stats.ms[CVO_KSTAT_ASSOC] += m_assoc;
      ctx->stats.launches[CVO_KSTAT_ASSOC] += 1;
      ctx->stats.ms[CVO_KSTAT_OVERFLOW] += m_ovf;
      ctx->stats.launches[CVO_KSTAT_OVERFLOW] += 1;
      ctx->stats.ms[CVO_KSTAT_BA_PAIR] += ms_pair;
      ctx->stats.launches[CVO_KSTAT_BA_PAIR] += pair_launches;
      ctx->stats.ms[CVO_KSTAT_BA_SOLVE] += ms_solve;
      ctx->stats.launches[CVO_KSTAT_BA_SOLVE] += solve_launches;
      le = hipGetLastError();
    } else {
      ba_iteration(L, st);
      le = hipGetLastError();
    }
    if (le != hipSuccess) {
      status = hip_check(ctx, le, "BA iteration launch");
      break;
    }
    // BaDev::iter and BaDev::done are adjacent
    hipError_t me = hipMemcpyAsync((void*)flag, &L.ba->iter, sizeof(int32_t) * 2, hipMemcpyDeviceToHost, st);
    if (me == hipSuccess) me = hipStreamSynchronize(st);
    if (me != hipSuccess) {
      status = hip_check(ctx, me, "BA flag readback");
      break;
    }
    const auto ti1 = std::chrono::steady_clock::now();
    if (per_iter_seconds && it < max_iter_records) per_iter_seconds[it] = std::chrono::duration<double>(ti1 - ti0).count();
    if (flag[1]) break;
  }
  if (use_graph) {
    (void)hipGraphExecDestroy(exec);
    (void)hipGraphDestroy(graph);
  }
  if (status != CVO_OK) return status;
  BaDev* out = new BaDev;
  const cvo_status re = read_back(ctx, out, L.ba, sizeof(BaDev));
  if (re != CVO_OK) {
    delete out;
    return re;
  }
  for (int f = 0; f < n_frames; ++f)
    for (int i = 0; i < 12; ++i) poses[12 * f + i] = out->X[12 * f + i];
  if (iters) *iters = out->iter;
  ctx->ba_last_accepted = out->accepted_total;
  ctx->ba_last_evals = out->evals_total;
  delete out;
  part_holder.release();  // the exports need the room
  // with multiframe_max_iters > 0 the first outer iteration associates
  const bool any_pass = p.multiframe_max_iters > 0;
  // each edge's pairs of the last association pass (BinaryStateGPU::
  // export_association, IRLS_State_GPU.cu:345-351; CvoGPU.cu:1990-1996)
  if (per_edge && any_pass)
    for (int e = 0; e < n_edges; ++e)
      CVO_TRY(export_problem(ctx, L.probs + e, frames[edges[2 * e]]->n, frames[edges[2 * e + 1]]->n, &per_edge[e]));
  if (seconds) *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t_start).count();
  return CVO_OK;
}
