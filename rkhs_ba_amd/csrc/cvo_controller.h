// The device controller of a registration: step length, pose update, indicator
// windows, lengthscale and the next pass's shape, on a ProblemState.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "cvo_device.h"
#include "cvo_internal.h"

namespace cvo {

// ---------------------------------------------------------------------------
// Device controller pieces (FP64)
// ---------------------------------------------------------------------------

// Real roots of a s^3 + b s^2 + c s + d by the trigonometric / Cardano closed
// form with two Newton polish steps; complex pairs report their imaginary part
// for the |imag| < 1e-5 rule of compute_step_size (CvoGPU.cu:513-519).
__device__ inline void cubic_solve(double a, double b, double c, double d, double re[3], double im[3]) {
  const double nan = __longlong_as_double(0x7ff8000000000000ll);
  re[0] = re[1] = re[2] = nan;
  im[0] = im[1] = im[2] = 0.0;
  if (!(a != 0.0)) return;
  const double p2 = b / a, p1 = c / a, p0 = d / a;
  if (!isfinite(p2) || !isfinite(p1) || !isfinite(p0)) return;
  const double sh = p2 / 3.0;
  const double p = p1 - p2 * sh;
  const double q = 2.0 * sh * sh * sh - sh * p1 + p0;
  const double disc = 0.25 * q * q + p * p * p / 27.0;
  auto polish = [&](double s) {
    for (int it = 0; it < 2; ++it) {
      double f = ((s + p2) * s + p1) * s + p0;
      double df = (3.0 * s + 2.0 * p2) * s + p1;
      if (df == 0.0) break;
      double ns = s - f / df;
      if (!isfinite(ns)) break;
      s = ns;
    }
    return s;
  };
  if (disc > 0.0) {
    const double sq = sqrt(disc);
    const double u = cbrt(-0.5 * q + (q > 0 ? -sq : sq));
    const double t = (u != 0.0) ? u - p / (3.0 * u) : 0.0;
    re[0] = polish(t - sh);
    const double ci = sqrt(fmax(0.75 * t * t + p, 0.0));
    re[1] = re[2] = -0.5 * t - sh;
    im[1] = ci;
    im[2] = -ci;
  } else if (p == 0.0) {
    re[0] = re[1] = re[2] = -sh;
  } else {
    const double m = 2.0 * sqrt(-p / 3.0);
    double arg = 3.0 * q / (p * m);
    arg = fmin(1.0, fmax(-1.0, arg));
    const double th = acos(arg) / 3.0;
    for (int k = 0; k < 3; ++k) re[k] = polish(m * cos(th - 2.0943951023931954923 * k) - sh);
  }
}

__device__ inline double select_step_dev(const KConsts& kc, const double bcde[4]) {
  double re[3], im[3];
  cubic_solve(4.0 * bcde[3], 3.0 * bcde[2], 2.0 * bcde[1], bcde[0], re, im);
  double temp = 1.7976931348623157e308;
  for (int i = 0; i < 3; ++i)
    if (re[i] > 0 && re[i] < temp && fabs(im[i]) < 1e-5) temp = re[i];
  if (temp > (double)kc.max_step) return (double)kc.max_step;
  if (temp < (double)kc.min_step) return (double)kc.min_step;
  return temp;
}

// A_sparsity_indicator_ell_update (CvoGPU.cu:547-665): two FIFO windows with
// float sums; ring buffers of modulus W+1.
__device__ inline bool indicator_update(ProblemState* st, float ind, int W, float thr) {
  const int cap = W + 1;
  bool dec = false;
  if (st->qs_size < W) {
    st->qs[(st->qs_head + st->qs_size) % cap] = ind;
    st->qs_size++;
    st->ss += ind;
  }
  if (st->qs_size >= W && st->qe_size < W) {
    st->qe[(st->qe_head + st->qe_size) % cap] = ind;
    st->qe_size++;
    st->se += ind;
  }
  if (st->qs_size >= W && st->qe_size >= W) {
    const float ratio = st->se / st->ss;
    if (ratio > 1.0f - thr && ratio < 1.0f + thr) {
      dec = true;
      st->qs_head = st->qs_size = st->qe_head = st->qe_size = 0;
      st->ss = 0.0f;
      st->se = 0.0f;
    } else {
      const float f = st->qe[st->qe_head];
      st->se -= f;
      st->ss += f;
      st->qs[(st->qs_head + st->qs_size) % cap] = f;
      st->qs_size++;
      st->qe_head = (st->qe_head + 1) % cap;
      st->qe_size--;
      st->ss -= st->qs[st->qs_head];
      st->qs_head = (st->qs_head + 1) % cap;
      st->qs_size--;
      st->qe[(st->qe_head + st->qe_size) % cap] = ind;
      st->qe_size++;
      st->se += ind;
    }
  }
  return dec;
}

// Float maps of the next iteration from the FP64 pose: target map [R^T, -R^T T]
// (update_tf, CvoGPU.cu:98-130) and the query map (R, T).
__device__ inline void set_maps(ProblemState* st) {
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < 3; ++j) {
      st->A[i * 3 + j] = (float)st->R[j * 3 + i];
      st->Rq[i * 3 + j] = (float)st->R[i * 3 + j];
    }
    st->b[i] = (float)(-(st->R[0 * 3 + i] * st->T[0] + st->R[1 * 3 + i] * st->T[1] + st->R[2 * 3 + i] * st->T[2]));
    st->Tq[i] = (float)st->T[i];
  }
}

__device__ inline int choose_level_tab(const float* h, int n_levels, float r_need) {
  int L = 0;
  for (int l = 0; l < n_levels; ++l)
    if (h[l] >= r_need) L = l;
  return L;
}

__device__ inline float needed_radius(const KConsts& kc, const ProblemState* st, float ell) {
  float tq = fmaxf(fabsf(st->Tq[0]), fmaxf(fabsf(st->Tq[1]), fabsf(st->Tq[2])));
  return kc.rq_coef * ell * (1.0f + kc.max_src_norm / 500.0f) * 1.0001f + 1e-4f * (1.0f + kc.max_src_norm + tq) + 1e-6f;
}

// Lanes per row and grid level of the next association pass at lengthscale
// ell (the level table given as cell sizes or as the grid).
__device__ inline void set_level(ProblemState* st, const KConsts& kc, float ell, const float* level_h, int n_levels) {
  const bool big = policy_big(kc.pol, ell);
  st->group = big ? kc.pol.group_big : kc.pol.group_small;
  st->level = choose_level_tab(level_h, n_levels,
                               needed_radius(kc, st, ell) * (big ? kc.pol.scale_big : kc.pol.scale_small));
}

__device__ inline void set_level(ProblemState* st, const KConsts& kc, float ell, const GridDev* grid) {
  const bool big = policy_big(kc.pol, ell);
  st->group = big ? kc.pol.group_big : kc.pol.group_small;
  st->level = choose_level(grid, needed_radius(kc, st, ell) * (big ? kc.pol.scale_big : kc.pol.scale_small));
}

__device__ inline double apply_step(ProblemState* st, const KConsts& kc, const double xi[6], const float xf[6],
                             double& step);

// One controller step of align_impl (CvoGPU.cu:1342-1433), FP64 pose state.
__device__ __forceinline__ void controller(ProblemState* st, const KConsts& kc, cvo_iter_record* trace,
                                           int trace_cap, int n_src, const float* level_h, int n_levels) {
  cvo_iter_record rec;
  const int k = st->iter;
  double fl[6];
  double n2 = 0.0;
  for (int c = 0; c < 6; ++c) {
    fl[c] = st->flow[c];
    n2 += fl[c] * fl[c];
  }
  const double nrm = sqrt(n2);
  double xi[6];
  for (int c = 0; c < 6; ++c) xi[c] = n2 > 0.0 ? fl[c] / nrm : fl[c];
  float xf[6];
  for (int c = 0; c < 6; ++c) xf[c] = (float)xi[c];
  const double nw = sqrt((double)xf[0] * xf[0] + (double)xf[1] * xf[1] + (double)xf[2] * xf[2]);
  const double nv = sqrt((double)xf[3] * xf[3] + (double)xf[4] * xf[4] + (double)xf[5] * xf[5]);
  rec.ell = st->ell;
  rec.nnz = (int32_t)st->nnz;
  rec.max_row = (int32_t)st->max_row;
  rec.num_neighbors = st->K;
  rec.flow_norm = (float)nrm;
  rec.step = 0.0f;
  rec.dist = 0.0f;
  rec.ip = (float)((double)st->nnz / sqrt((double)kc.n_src_f * (double)kc.n_tgt_f));
  if (nw < (double)kc.eps && nv < (double)kc.eps) {
    st->ret = (nw < 1e-8 && nv < 1e-8) ? -1 : 0;
    st->done = 1;
    st->iters_out = k;
    if (trace && k < trace_cap) trace[k] = rec;
    return;
  }
  double step = select_step_dev(kc, st->bcde);
  const double dist = apply_step(st, kc, xi, xf, step);
  st->step = step;
  st->dist = dist;
  rec.step = (float)step;
  rec.dist = (float)dist;
  const bool dec = indicator_update(st, rec.ip, kc.window, kc.ind_thr);
  if (trace && k < trace_cap) trace[k] = rec;
  set_maps(st);
  if (dist < (double)kc.eps_2) {
    st->done = 1;
    st->iters_out = k;
    return;
  }
  if (k > kc.ell_decay_start && dec) {
    float e = st->ell * kc.ell_decay_rate;
    if (e < kc.ell_min) e = kc.ell_min;
    st->ell = e;
  }
  if (kc.knn > 0) {
    // K nearest: the mean stored row rounded up times is_using_kdtree, at
    // most KDTREE_K_SIZE (CvoGPU.cu:1416-1417); zero stays zero
    const int mean = (int)ceil((double)st->nnz / (double)n_src);
    st->K = min(kKnnMaxK, mean * kc.knn);
  } else {
    st->K = min(kc.nn_max, (int)((double)st->max_row * 1.2));
    if (st->K < 1) st->K = 1;
  }
  st->iter = k + 1;
  if (st->iter >= kc.max_iter) {
    st->done = 1;
    st->iters_out = kc.max_iter;
  }
  set_level(st, kc, st->ell, level_h, n_levels);
  st->n_overflow = 0;
}

// Pose update by exp(step xi) (CvoGPU.cu:1362-1379): FP64 by default, or the
// reference's float arithmetic (float step, FP32 Exp_SEK3, pose products in
// double rounded to float).  Returns the step's SE(3) distance; step is
// rounded to float in the reference mode.
__device__ inline double apply_step(ProblemState* st, const KConsts& kc, const double xi[6], const float xf[6],
                             double& step) {
  double dR[9], dT[3];
  double dist;
  if (kc.mirror_pose) {
    // the reference's float pose arithmetic: float step, FP32 Exp_SEK3, the
    // pose products in double rounded to float (CvoGPU.cu:1289-1341)
    step = (double)(float)step;
    float e[12];
    exp_sek3_f32(xf, (float)step, e);
    for (int r = 0; r < 3; ++r) {
      for (int c = 0; c < 3; ++c) dR[r * 3 + c] = (double)e[r * 4 + c];
      dT[r] = (double)e[r * 4 + 3];
    }
    double Rn[9], Tn[3];
    for (int r = 0; r < 3; ++r) {
      Tn[r] = (double)(float)(st->R[r * 3 + 0] * dT[0] + st->R[r * 3 + 1] * dT[1] + st->R[r * 3 + 2] * dT[2] + st->T[r]);
      for (int c = 0; c < 3; ++c)
        Rn[r * 3 + c] = (double)(float)(st->R[r * 3 + 0] * dR[0 * 3 + c] + st->R[r * 3 + 1] * dR[1 * 3 + c] +
                                        st->R[r * 3 + 2] * dR[2 * 3 + c]);
    }
    for (int i = 0; i < 9; ++i) st->R[i] = Rn[i];
    for (int i = 0; i < 3; ++i) st->T[i] = Tn[i];
    dist = se3_log_norm(dR, dT);
  } else {
    se3_exp(xi, step, dR, dT);
    double Rn[9], Tn[3];
    for (int r = 0; r < 3; ++r) {
      Tn[r] = st->T[r] + st->R[r * 3 + 0] * dT[0] + st->R[r * 3 + 1] * dT[1] + st->R[r * 3 + 2] * dT[2];
      for (int c = 0; c < 3; ++c)
        Rn[r * 3 + c] = st->R[r * 3 + 0] * dR[0 * 3 + c] + st->R[r * 3 + 1] * dR[1 * 3 + c] + st->R[r * 3 + 2] * dR[2 * 3 + c];
    }
    for (int i = 0; i < 9; ++i) st->R[i] = Rn[i];
    for (int i = 0; i < 3; ++i) st->T[i] = Tn[i];
    // ||log(exp(step xi))|| = step ||xi|| exactly while the rotation angle
    // step*|w| stays below pi; the general log otherwise
    const double wn = sqrt(xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2]);
    const double xn = sqrt(xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2] + xi[3] * xi[3] + xi[4] * xi[4] + xi[5] * xi[5]);
    dist = (step * wn < 3.0) ? step * xn : se3_log_norm(dR, dT);
  }
  return dist;
}

// Step length of the adaptive-lengthscale loop (AdaptiveCvoGPU.cu:1006-1075):
// the cubic's coefficients rounded to float, its smallest positive real root,
// min_step when there is none, at most 0.8.
__device__ inline double select_step_adaptive(const KConsts& kc, const double bcde[4]) {
  double re[3], im[3];
  cubic_solve((double)(4.0f * (float)bcde[3]), (double)(3.0f * (float)bcde[2]), (double)(2.0f * (float)bcde[1]),
              (double)(float)bcde[0], re, im);
  double temp = 1.7976931348623157e308;
  for (int i = 0; i < 3; ++i)
    if (re[i] > 0 && re[i] < temp && im[i] == 0.0) temp = re[i];
  double step = temp == 1.7976931348623157e308 ? (double)kc.min_step : (double)(float)temp;
  return step > 0.8 ? 0.8 : step;
}

// One controller step of AdaptiveCvoGPU::align (AdaptiveCvoGPU.cu:1117-1205):
// unnormalised flow (omega / c, v / d), stop when both parts are below eps,
// exp(step xi), stop when the step's distance is below eps_2, then the
// lengthscale moves against its gradient
//   dl = (2/l^3 sum_A -a |y-x|^2 + 1/l^3 sum_Axx a |x'-x|^2 + 1/l^3 sum_Ayy a |y'-y|^2)
//        / (nnz(Axx) + nnz(Ayy) - 2 nnz(A))            (:445-890, unsigned count)
//   l <- l - dl_step dl; past ell_max both shrink to 0.7 ell_max; at least ell_min.
// The source and target self-association totals come from sx / sy
// (their passes ran with this one; st->ip holds sum(a |y-x|^2)).
__device__ __forceinline__ void controller_adaptive(ProblemState* st, const ProblemState* sx, const ProblemState* sy,
                                                    const KConsts& kc, cvo_iter_record* trace, int trace_cap,
                                                    const float* level_h, int n_levels) {
  cvo_iter_record rec;
  const int k = st->iter;
  float xf[6];
  double xi[6];
  for (int c = 0; c < 6; ++c) {
    xf[c] = (float)st->flow[c];
    xi[c] = (double)xf[c];
  }
  const double nw = sqrt(xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2]);
  const double nv = sqrt(xi[3] * xi[3] + xi[4] * xi[4] + xi[5] * xi[5]);
  rec.ell = st->ell;
  rec.nnz = (int32_t)st->nnz;
  rec.max_row = (int32_t)st->max_row;
  rec.num_neighbors = st->K;
  rec.flow_norm = (float)sqrt(nw * nw + nv * nv);
  rec.step = 0.0f;
  rec.dist = 0.0f;
  rec.ip = (float)((double)st->nnz / sqrt((double)kc.n_src_f * (double)kc.n_tgt_f));
  if (nw < (double)kc.eps && nv < (double)kc.eps) {
    st->ret = (nw < 1e-8 && nv < 1e-8) ? -1 : 0;
    st->done = 1;
    st->iters_out = k;
    if (trace && k < trace_cap) trace[k] = rec;
    return;
  }
  double step = select_step_adaptive(kc, st->bcde);
  const double dist = apply_step(st, kc, xi, xf, step);
  st->step = step;
  st->dist = dist;
  rec.step = (float)step;
  rec.dist = (float)dist;
  if (trace && k < trace_cap) trace[k] = rec;
  set_maps(st);
  if (dist < (double)kc.eps_2) {
    st->done = 1;
    st->iters_out = k;
    return;
  }
  const float l3 = st->ell * st->ell * st->ell;
  const float dl_a = (float)((-2.0 * st->ip + sx->ip) / (double)l3);
  const float dl_yy = (float)(sy->ip / (double)l3);
  const uint32_t denom = (uint32_t)sx->nnz + (uint32_t)sy->nnz - 2u * (uint32_t)st->nnz;
  const double dl = (double)(dl_a + dl_yy) / (double)denom;
  st->dl = dl;
  float ell = (float)((double)st->ell - kc.dl_step * dl);
  if (ell >= st->ell_max) {
    ell = (float)((double)st->ell_max * 0.7);
    st->ell_max = (float)((double)st->ell_max * 0.7);
  }
  st->ell = ell < kc.ell_min ? kc.ell_min : ell;
  st->iter = k + 1;
  if (st->iter >= kc.max_iter) {
    st->done = 1;
    st->iters_out = kc.max_iter;
  }
  set_level(st, kc, st->ell, level_h, n_levels);
  st->n_overflow = 0;
}

// A self-association problem (q = 1 source, 2 target) follows the registration
// problem of an adaptive-lengthscale run: lengthscale, iteration, done flag; the
// target problem's points move with the target map.
__device__ inline void adaptive_follow(ProblemState* st, const ProblemState* s0, int q, const KConsts& kc,
                                       const float* level_h, int n_levels) {
  st->ell = s0->ell;
  st->K = s0->K;
  st->iter = s0->iter;
  st->done = s0->done;
  st->n_overflow = 0;
  for (int i = 0; i < 9; ++i) {
    const float e = (i % 4 == 0) ? 1.0f : 0.0f;
    st->A[i] = q == 2 ? s0->A[i] : e;
    st->As[i] = q == 2 ? s0->A[i] : e;
    st->Rq[i] = q == 2 ? s0->Rq[i] : e;
  }
  for (int i = 0; i < 3; ++i) {
    st->b[i] = q == 2 ? s0->b[i] : 0.0f;
    st->bs[i] = q == 2 ? s0->b[i] : 0.0f;
    st->Tq[i] = q == 2 ? s0->Tq[i] : 0.0f;
  }
  st->has_src_xf = q == 2 ? 1 : 0;
  set_level(st, kc, st->ell, level_h, n_levels);
}

}  // namespace cvo
