// Association rows, capped rows and step terms: the device code of a
// registration's passes, shared by the pass kernels and the resident loop.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "cvo_ball.h"
#include "cvo_device.h"
#include "cvo_internal.h"

namespace cvo {

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------

// Workgroups are dispatched to the eight XCDs round robin by id (XCD = id % 8).
// This maps a dispatch id to a logical block so that every XCD takes one
// contiguous range of logical blocks: spatially sorted rows whose overlapping
// target neighbourhoods its own L2 then serves.  A bijection of [0, nblk).
__device__ __forceinline__ int xcd_block(int bid, int nblk) {
  const int q = nblk >> 3, r = nblk & 7;
  const int x = bid & 7, k = bid >> 3;
  return (x < r) ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
}

// Cross-block publication without cache maintenance.  Partials are written
// with device-scope stores (sc1: written through to the device coherence
// point) by lanes of wave 0, which then waits for its stores (vmcnt(0))
// before lane 0 counts the block in with a device-scope atomic; the block
// that counts last reads the partials with device-scope loads.  An agent
// fence would instead write back and invalidate the whole XCD L2 in every
// block, which costs the association kernel its cached target neighbourhoods.
__device__ __forceinline__ void st_dev(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_dev(double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t ld_dev(uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t count_in(uint32_t* counter) {
  return __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima), between two
// compiler-only fences: the builtin orders the hardware, the fences keep the
// compiler from moving the partial stores past it or the completion atomic
// before it (neither fence emits an instruction or a cache operation).
__device__ __forceinline__ void wait_stores() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Exact evaluation of a pair's kernel value with FP64 exponentials rounded to
// float, the reference's rounding points (CvoGPU.cu:1020-1054).  Used only for
// pairs whose fast FP32 value lies within 2e-5 relative of sp_thres, so the
// stored set equals the reference's.
static __device__ __noinline__ float exact_value(float sigma2, float c_sigma2, float s_sigma2, float c2, float s_ell,
                                         int use_geo, int use_col, int use_sem, float d2, float l, float d2c,
                                         float d2s, float geo_sim) {
  float k = 1.0f, ck = 1.0f, sk = 1.0f;
  if (use_geo) k = (float)((double)sigma2 * exp((double)(-d2) / (2.0 * (double)l * (double)l)));
  if (use_col) ck = (float)((double)c_sigma2 * exp((double)(-d2c) / (2.0 * (double)c2)));
  if (use_sem) sk = (float)((double)s_sigma2 * exp((double)(-d2s) / (2.0 * (double)s_ell * (double)s_ell)));
  return ck * k * sk * geo_sim;
}

__device__ __forceinline__ float geo_similarity(const float* ga, const float* gb) {
  float n2a = fmaf(ga[1], ga[1], ga[0] * ga[0]);
  float n2b = fmaf(gb[1], gb[1], gb[0] * gb[0]);
  float dab = fmaf(ga[1], gb[1], ga[0] * gb[0]);
  return dab * dab / (n2a * n2b);
}

// |y - x|^2 with the association's FMA order.
__device__ __forceinline__ float sq_dist(float x0, float x1, float x2, float y0, float y1, float y2) {
  const float dx = y0 - x0, dy = y1 - x1, dz = y2 - x2;
  return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// Locate the problem of a flat block index.
__device__ __forceinline__ int find_problem(const AssocProblem* probs, int n_probs, int blk) {
  int lo = 0, hi = n_probs - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (probs[mid].block_begin <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// Association + fused flow
// ---------------------------------------------------------------------------

// Loads a scalar feature (compile-time or runtime dimension).
template <int N>
struct Dim {
  __device__ static constexpr int get(int) { return N; }
};
template <>
struct Dim<-1> {
  __device__ static int get(int rt) { return rt; }
};

// Float maps of one iteration, loaded once per block from the problem state.
struct Maps {
  float A[9], b[3];    // target: y' = A y + b
  float Rq[9], Tq[3];  // query into the target frame
  float As[9], bs[3];  // source map
  bool src_xf;
};

__device__ __forceinline__ void load_maps(const ProblemState* st, Maps& m) {
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    m.A[i] = st->A[i];
    m.Rq[i] = st->Rq[i];
    m.As[i] = st->As[i];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    m.b[i] = st->b[i];
    m.Tq[i] = st->Tq[i];
    m.bs[i] = st->bs[i];
  }
  m.src_xf = st->has_src_xf != 0;
}

// Scalars of the exact path (passed by value: no private copy of KConsts).
struct ExactK {
  float sigma2, c_sigma2, s_sigma2, c2, s_ell;
  int use_geo, use_col, use_sem;
};

__device__ __forceinline__ ExactK exact_consts(const KConsts& kc) {
  ExactK e;
  e.sigma2 = kc.sigma2;
  e.c_sigma2 = kc.c_sigma2;
  e.s_sigma2 = kc.s_sigma2;
  e.c2 = kc.c2;
  e.s_ell = kc.s_ell;
  e.use_geo = kc.use_geo && !kc.no_geo_factor;
  e.use_col = kc.use_col;
  e.use_sem = kc.use_sem;
  return e;
}

// The kernel value of a candidate pair: gates, then the product kernel.
// Returns false when a gate rejects or a <= sp_thres.  gmin: the geometric
// type similarity below which a pair is rejected (0.01 in fill_in_A_mat_gpu,
// CvoGPU.cu:1015; 0.001 in fill_in_A_mat_cukdtree, :898).
template <int FC, int KC>
__device__ __forceinline__ bool pair_kernel(const KConsts& kc, const ExactK& ek, float x0, float x1, float x2,
                                            float y0, float y1, float y2, float d2t, float qg, float l,
                                            const float* xf, const float* yf, const float* xs, const float* ys,
                                            const float* xg, const float* yg, float& a, float gmin = 0.01f) {
  const float dx = y0 - x0, dy = y1 - x1, dz = y2 - x2;
  const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  if (kc.use_geo && !(d2 < d2t)) return false;
  float geo_sim = 1.0f;
  if (kc.use_gtype) {
    // yg always addresses the target cloud's type vectors in global memory
    const float ygl[2] = {ld_global(yg), ld_global(yg + 1)};
    geo_sim = geo_similarity(xg, ygl);
    if (geo_sim < gmin) return false;
  }
  float d2c = 0.0f, d2s = 0.0f;
  if (FC != 0) {
    const int F = Dim<FC>::get(kc.F);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      float t = xf[f] - yf[f];
      d2c = fmaf(t, t, d2c);
    }
    if (!(d2c < kc.d2_c_thres)) return false;
  }
  if (KC != 0) {
    const int KS = Dim<KC>::get(kc.Ks);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      float t = xs[k] - ys[k];
      d2s = fmaf(t, t, d2s);
    }
    if (!(d2s < kc.d2_s_thres)) return false;
  }
  float ex = (kc.use_geo && !kc.no_geo_factor) ? d2 * qg : 0.0f;
  if (FC != 0) ex = fmaf(d2c, kc.q_c, ex);
  if (KC != 0) ex = fmaf(d2s, kc.q_s, ex);
  a = kc.amp * expf(-ex) * geo_sim;
  if (fabsf(a - kc.sp) <= 2e-5f * kc.sp)
    a = exact_value(ek.sigma2, ek.c_sigma2, ek.s_sigma2, ek.c2, ek.s_ell, ek.use_geo, ek.use_col, ek.use_sem, d2, l,
                    d2c, d2s, geo_sim);
  return a > kc.sp;
}

// Stores one kept pair of row r in slot `slot`: the bundle adjustment keeps
// the target's own coordinates and a at the iteration's row stride K (and,
// when asked, the target's sorted position for an association export);
// the other modes keep (sorted target position, a) at the allocated stride,
// unless the pass only sums (no pair array).
// NOBA: the launch never carries a bundle-adjustment problem (single-problem
// kernels), so that store is compiled out.
template <bool NOBA = false>
__device__ __forceinline__ void store_pair(const AssocProblem& P, int mode, int r, uint32_t K, uint32_t slot,
                                           uint32_t pidx, const float4& y4, float a) {
  if (!NOBA && mode == MODE_BA) {
    st_global(P.pairs4 + (size_t)r * K + slot, make_float4(y4.x, y4.y, y4.z, a));
    if (P.pair_ids) st_global(P.pair_ids + (size_t)r * K + slot, pidx);
  } else if (P.pairs) {
    st_global(P.pairs + (size_t)r * P.cap_alloc + slot, make_uint2(pidx, __float_as_uint(a)));
  }
}

// A row's constants at one lengthscale: its own lengthscale, the distance
// gate, the factor of d2 in the exponent, and the gate's radius with the margin
// of the query box.  x: the row's (mapped) point.
struct RowConsts {
  float l, d2t, qg, r;
};
__device__ __forceinline__ RowConsts row_consts(const KConsts& kc, bool own_ell, float ell, float x0, float x1,
                                                float x2) {
  RowConsts c;
  c.l = own_ell ? range_ell(ell, x0, x1, x2) : ell;
  c.d2t = (float)(-2.0 * (double)c.l * (double)c.l * (double)kc.lg);
  c.qg = (float)(1.0 / (2.0 * (double)c.l * (double)c.l));
  c.r = sqrtf(c.d2t) * 1.001f;
  return c;
}

struct RowResult {
  double acc[7];  // omega(3), v(3), ip
  uint32_t stored;
  bool overflow;
};

// One row (source point x4, features xf, class vector xs) handled by a group
// of G lanes.  FC/KC: color/semantic dimension when the
// gate is on (0 off, -1 runtime).  MODE_ALIGN accumulates the flow, MODE_IP and
// MODE_BA only the sum of a.
template <int FC, int KC, int G, bool NOBA>
__device__ __forceinline__ void assoc_row(const AssocProblem& P, const KConsts& kc, const ExactK& ek,
                                          const GridLevel& GL, const Maps& mp, int r, int g, int mode, float ell,
                                          int K, const float4& x4, const float* xf, const float* xs, RowResult& out,
                                          const RowConsts* rc = nullptr) {
#pragma unroll
  for (int c = 0; c < 7; ++c) out.acc[c] = 0.0;
  out.stored = 0;
  out.overflow = false;
  const uint32_t Ku = (uint32_t)K;
  if (!kc.use_geo) {
    // no distance gate: every target is a candidate, so the row takes the
    // exact full scan of the capped-row kernel
    out.stored = Ku + 1u;
    out.overflow = true;
    return;
  }
  const int F = Dim<FC>::get(kc.F);
  const int KS = Dim<KC>::get(kc.Ks);
  float x0 = x4.x, x1 = x4.y, x2 = x4.z;
  if (mp.src_xf) {
    float t0, t1, t2;
    affine3(mp.As, mp.bs, x0, x1, x2, t0, t1, t2);
    x0 = t0; x1 = t1; x2 = t2;
  }
  // the adaptive-lengthscale association uses ell as is (AdaptiveCvoGPU.cu:281)
  const RowConsts rk = rc ? *rc : row_consts(kc, !kc.fixed_ell, ell, x0, x1, x2);
  const float l = rk.l, d2t = rk.d2t, qg = rk.qg;
  float xg[2] = {0.0f, 0.0f};
  if (kc.use_gtype) {
    xg[0] = ld_global(P.src_geo + 2 * (size_t)r);
    xg[1] = ld_global(P.src_geo + 2 * (size_t)r + 1);
  }
  // query box in the target frame
  float q0, q1, q2;
  affine3(mp.Rq, mp.Tq, x0, x1, x2, q0, q1, q2);
  const float rq = rk.r + 1e-4f * (1.0f + fmaxf(fabsf(q0), fmaxf(fabsf(q1), fabsf(q2))));
  int lo0 = cell_floor((q0 - rq - GL.ox) * GL.inv_h, GL.nx), hi0 = cell_floor((q0 + rq - GL.ox) * GL.inv_h, GL.nx);
  int lo1 = cell_floor((q1 - rq - GL.oy) * GL.inv_h, GL.ny), hi1 = cell_floor((q1 + rq - GL.oy) * GL.inv_h, GL.ny);
  int lo2 = cell_floor((q2 - rq - GL.oz) * GL.inv_h, GL.nz), hi2 = cell_floor((q2 + rq - GL.oz) * GL.inv_h, GL.nz);
  int nruns = 0, span1 = 0;
  if (!(hi0 < 0 || lo0 >= GL.nx || hi1 < 0 || lo1 >= GL.ny || hi2 < 0 || lo2 >= GL.nz)) {
    lo0 = max(lo0, 0); hi0 = min(hi0, GL.nx - 1);
    lo1 = max(lo1, 0); hi1 = min(hi1, GL.ny - 1);
    lo2 = max(lo2, 0); hi2 = min(hi2, GL.nz - 1);
    span1 = hi1 - lo1 + 1;
    nruns = span1 * (hi2 - lo2 + 1);
  }
  uint32_t stored = 0;
  bool stop = false;
  // batched launches (bundle adjustment, multi-start): a run's cells beyond
  // the query radius hold no passing target, so the run is clipped to the
  // ball's chord over its (y, z) cell square, or skipped; the slack covers
  // the float rounding of the points' cell assignment, and rq itself exceeds
  // the distance gate's radius, so no passing target is lost and the passing
  // targets keep their enumeration order.  (Single-problem launches do not
  // clip: their fine cells leave little to cut, and the extra arithmetic on
  // the row's dependent chain costs more.)
  constexpr bool CLIP = !NOBA;
  const float rq2 = rq * rq, slack = 1e-3f * GL.h;
  (void)rq2;
  (void)slack;
  for (int rbase = 0; rbase < nruns && !stop; rbase += G) {
    const int myrun = rbase + g;
    uint32_t rs = 0, rl = 0;
    if (myrun < nruns) {
      const int iz = myrun / span1, iy = myrun - iz * span1;
      if constexpr (CLIP) {
        const int cy = lo1 + iy, cz = lo2 + iz;
        const float ys = GL.oy + (float)cy * GL.h, zs = GL.oz + (float)cz * GL.h;
        const float dy = fmaxf(0.0f, fmaxf(ys - q1, q1 - (ys + GL.h)) - slack);
        const float dz = fmaxf(0.0f, fmaxf(zs - q2, q2 - (zs + GL.h)) - slack);
        const float rem = rq2 - (dy * dy + dz * dz);
        if (rem >= 0.0f) {  // else the run lies beyond the radius
          const float ch = sqrtf(rem) + slack;
          const int lo = max(lo0, cell_floor((q0 - ch - GL.ox) * GL.inv_h, GL.nx));
          const int hi = min(hi0, cell_floor((q0 + ch - GL.ox) * GL.inv_h, GL.nx));
          if (lo <= hi) {
            const uint32_t c0 = ((uint32_t)cz * (uint32_t)GL.ny + (uint32_t)cy) * (uint32_t)GL.nx + (uint32_t)lo;
            rs = ld_global(GL.cell_start + c0);
            rl = ld_global(GL.cell_start + c0 + (uint32_t)(hi - lo) + 1u) - rs;
          }
        }
      } else {
        const uint32_t c0 =
            ((uint32_t)(lo2 + iz) * (uint32_t)GL.ny + (uint32_t)(lo1 + iy)) * (uint32_t)GL.nx + (uint32_t)lo0;
        rs = ld_global(GL.cell_start + c0);
        rl = ld_global(GL.cell_start + c0 + (uint32_t)(hi0 - lo0) + 1u) - rs;
      }
    }
    uint32_t incl = rl;
#pragma unroll
    for (int o = 1; o < G; o <<= 1) {
      uint32_t t = __shfl_up(incl, o, G);
      if (g >= o) incl += t;
    }
    const uint32_t total = __shfl(incl, G - 1, G);
    const uint32_t excl = incl - rl;
    for (uint32_t base = 0; base < total; base += G) {
      const uint32_t idx = base + (uint32_t)g;
      // the run holding candidate idx: the last run whose prefix is <= idx
      int kk = 0;
#pragma unroll
      for (int s = G / 2; s > 0; s >>= 1) {
        uint32_t e = __shfl(excl, kk + s, G);
        if (e <= idx) kk += s;
      }
      const uint32_t run_start = __shfl(rs, kk, G);
      const uint32_t run_excl = __shfl(excl, kk, G);
      bool pass = false;
      float a = 0.0f, y0 = 0.0f, y1 = 0.0f, y2 = 0.0f;
      uint32_t pidx = 0;
      float4 y4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (idx < total) {
        pidx = run_start + (idx - run_excl);
        y4 = ld_global(GL.pos + pidx);
        // with compile-time dimensions the candidate's features and class
        // vector are loaded together with its position, before the gates
        // that may not need them: one memory round trip instead of three
        float yfr[FC > 0 ? FC : 1], ysr[KC > 0 ? KC : 1];
        if (FC > 0) {
#pragma unroll
          for (int f = 0; f < (FC > 0 ? FC : 1); ++f) yfr[f] = ld_global(GL.feat + (size_t)pidx * F + f);
        }
        if (KC > 0) {
#pragma unroll
          for (int k = 0; k < (KC > 0 ? KC : 1); ++k) ysr[k] = ld_global(GL.sem + (size_t)pidx * KS + k);
        }
        affine3(mp.A, mp.b, y4.x, y4.y, y4.z, y0, y1, y2);
        pass = pair_kernel<FC, KC>(kc, ek, x0, x1, x2, y0, y1, y2, d2t, qg, l, xf,
                                   FC > 0 ? yfr : (FC != 0 ? GL.feat + (size_t)pidx * F : nullptr), xs,
                                   KC > 0 ? ysr : (KC != 0 ? GL.sem + (size_t)pidx * KS : nullptr), xg,
                                   kc.use_gtype ? GL.geo + 2 * (size_t)pidx : nullptr, a);
      }
      const uint64_t m = __ballot(pass);
      const auto gm = group_ballot<G>(m);
      const uint32_t slot = stored + group_count(gm & ((decltype(gm))(1ull << g) - 1u));
      if (pass && (slot < Ku || kc.uncapped)) {
        if (slot < Ku) store_pair<NOBA>(P, mode, r, Ku, slot, pidx, y4, a);
        if (mode == MODE_ALIGN) {
          const float c0 = x1 * y2 - x2 * y1, c1 = x2 * y0 - x0 * y2, c2 = x0 * y1 - x1 * y0;
          out.acc[0] += (double)(c0 * a);
          out.acc[1] += (double)(c1 * a);
          out.acc[2] += (double)(c2 * a);
          out.acc[3] += (double)((y0 - x0) * a);
          out.acc[4] += (double)((y1 - x1) * a);
          out.acc[5] += (double)((y2 - x2) * a);
        }
        out.acc[6] += (double)(kc.ip_ad2 ? sq_dist(x0, x1, x2, y0, y1, y2) * a : a);
      }
      stored += group_count(gm);
      if (stored > Ku && !kc.uncapped) {
        stop = true;
        break;
      }
    }
  }
  // uncapped: every passing pair is summed, the first K stored
  out.stored = kc.uncapped ? min(stored, Ku) : stored;
  out.overflow = stored > Ku && !kc.uncapped;
}

// ---------------------------------------------------------------------------
// K-nearest association (is_using_kdtree: se_kernel_kdtree, CvoGPU.cu:1104-1154,
// fill_in_A_mat_cukdtree :832-949).  A row's candidates are its K nearest
// targets, nearest first; each must then pass the gates, the distance gate at
// the fixed lengthscale (no range scaling, :863).  A target outside the
// distance gate's ball can never be stored, and a target inside it is among
// the K nearest exactly when fewer than K ball targets are nearer, so the
// selection runs over the ball alone.  Nearness is the key (float d2 bits,
// target id): ties by ascending id.  A row counts its ball targets; with more
// than K, a most-significant-digit radix select over the keys (8 bits a pass,
// one 256-bin LDS histogram per row) finds the K-th smallest key.  The last
// pass applies the gates to the selected targets and stores the passing ones.
// ---------------------------------------------------------------------------

template <int FC, int KC, int G>
__device__ __forceinline__ void knn_row(const AssocProblem& P, const KConsts& kc, const ExactK& ek,
                                        const GridLevel& GL, const Maps& mp, int r, int g, int mode, float ell, int K,
                                        const float4& x4, const float* xf, const float* xs, uint32_t* hist,
                                        RowResult& out, const RowConsts* rc = nullptr) {
#pragma unroll
  for (int c = 0; c < 7; ++c) out.acc[c] = 0.0;
  out.stored = 0;
  out.overflow = false;
  const uint32_t Ku = (uint32_t)max(K, 0);
  if (Ku == 0) return;
  const int F = Dim<FC>::get(kc.F);
  const int KS = Dim<KC>::get(kc.Ks);
  float x0 = x4.x, x1 = x4.y, x2 = x4.z;
  if (mp.src_xf) {
    float t0, t1, t2;
    affine3(mp.As, mp.bs, x0, x1, x2, t0, t1, t2);
    x0 = t0; x1 = t1; x2 = t2;
  }
  const RowConsts rk = rc ? *rc : row_consts(kc, false, ell, x0, x1, x2);
  const float l = rk.l, d2t = rk.d2t, qg = rk.qg;
  float xg[2] = {0.0f, 0.0f};
  if (kc.use_gtype) {
    xg[0] = ld_global(P.src_geo + 2 * (size_t)r);
    xg[1] = ld_global(P.src_geo + 2 * (size_t)r + 1);
  }
  float q0, q1, q2;
  affine3(mp.Rq, mp.Tq, x0, x1, x2, q0, q1, q2);
  const float rq = rk.r + 1e-4f * (1.0f + fmaxf(fabsf(q0), fmaxf(fabsf(q1), fabsf(q2))));
  const CellBox B = cell_box(GL, q0, q1, q2, rq);
  // key of a target, ~0 outside the ball (no ball key reaches it: d2 bits of
  // a finite d2 < d2t stay below 0x7f800000)
  auto key_of = [&](uint32_t pidx, float4& y4, float& y0, float& y1, float& y2) -> uint64_t {
    y4 = ld_global(GL.pos + pidx);
    affine3(mp.A, mp.b, y4.x, y4.y, y4.z, y0, y1, y2);
    const float dx = y0 - x0, dy = y1 - x1, dz = y2 - x2;
    const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    if (!(d2 < d2t)) return ~0ull;
    return ((uint64_t)__float_as_uint(d2) << 32) | (uint64_t)__float_as_uint(y4.w);
  };
  // (1)-(2) the K nearest of the ball: thr / tsh bound their keys
  uint64_t thr;
  int tsh;
  select_smallest<G>(
      [&](auto&& fn) { for_each_in_box<G>(GL, B, g, fn); }, g, Ku, hist,
      [&](uint32_t pidx) {
        float4 y4;
        float y0, y1, y2;
        return key_of(pidx, y4, y0, y1, y2);
      },
      thr, tsh);
  // (3) gates on the selected targets, stored in slots by ballot
  uint32_t stored = 0;
  for_each_in_box<G>(GL, B, g, [&](bool valid, uint32_t pidx) {
    bool pass = false;
    float a = 0.0f, y0 = 0.0f, y1 = 0.0f, y2 = 0.0f;
    float4 y4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid) {
      const uint64_t key = key_of(pidx, y4, y0, y1, y2);
      if (selected(key, thr, tsh)) {
        // compile-time dimensions: the target's features and class vector
        // loaded into registers through global-address loads
        float yfr[FC > 0 ? FC : 1], ysr[KC > 0 ? KC : 1];
        if (FC > 0) {
#pragma unroll
          for (int f = 0; f < (FC > 0 ? FC : 1); ++f) yfr[f] = ld_global(GL.feat + (size_t)pidx * F + f);
        }
        if (KC > 0) {
#pragma unroll
          for (int k = 0; k < (KC > 0 ? KC : 1); ++k) ysr[k] = ld_global(GL.sem + (size_t)pidx * KS + k);
        }
        pass = pair_kernel<FC, KC>(kc, ek, x0, x1, x2, y0, y1, y2, d2t, qg, l, xf,
                                   FC > 0 ? yfr : (FC != 0 ? GL.feat + (size_t)pidx * F : nullptr), xs,
                                   KC > 0 ? ysr : (KC != 0 ? GL.sem + (size_t)pidx * KS : nullptr), xg,
                                   kc.use_gtype ? GL.geo + 2 * (size_t)pidx : nullptr, a, 0.001f);
      }
    }
    const uint32_t gm = group_bits<G>(__ballot(pass));
    const uint32_t slot = stored + (uint32_t)__popc(gm & ((1u << g) - 1u));
    if (pass && slot < Ku) {
      store_pair(P, mode, r, Ku, slot, pidx, y4, a);
      if (mode == MODE_ALIGN) {
        const float c0 = x1 * y2 - x2 * y1, c1 = x2 * y0 - x0 * y2, c2 = x0 * y1 - x1 * y0;
        out.acc[0] += (double)(c0 * a);
        out.acc[1] += (double)(c1 * a);
        out.acc[2] += (double)(c2 * a);
        out.acc[3] += (double)((y0 - x0) * a);
        out.acc[4] += (double)((y1 - x1) * a);
        out.acc[5] += (double)((y2 - x2) * a);
      }
      out.acc[6] += (double)a;
    }
    stored += (uint32_t)__popc(gm);
  });
  out.stored = min(stored, Ku);
}

// A row whose passing pairs exceed the cap keeps the first K passing targets
// by ascending target index (CvoGPU.cu:994-996).  Every passing target lies
// in the distance gate's ball, so one wave finds them there: it counts the
// ball's passing targets and their index range, selects the K smallest
// indices by a most-significant-digit radix select (8 bits a pass, a 256-bin
// LDS histogram), then stores exactly those.  acc: the lane's share of the
// row's flow and ip; returns the stored count.
template <int FC, int KC>
__device__ inline uint32_t capped_row_ball(const AssocProblem& P, const KConsts& kc, const ExactK& ek,
                                           const GridLevel& GL, const Maps& mp, int r, float ell, uint32_t K,
                                           uint32_t* hist, double acc[7], int mode) {
  const int g = threadIdx.x & 63;
  const int F = Dim<FC>::get(kc.F);
  const int KS = Dim<KC>::get(kc.Ks);
  float4 x4 = ld_global(P.src_pos + r);
  float x0 = x4.x, x1 = x4.y, x2 = x4.z;
  if (mp.src_xf) {
    float t0, t1, t2;
    affine3(mp.As, mp.bs, x0, x1, x2, t0, t1, t2);
    x0 = t0; x1 = t1; x2 = t2;
  }
  const float l = kc.fixed_ell ? ell : range_ell(ell, x0, x1, x2);
  const float d2t = (float)(-2.0 * (double)l * (double)l * (double)kc.lg);
  const float qg = (float)(1.0 / (2.0 * (double)l * (double)l));
  // with compile-time dimensions the row's and each candidate's features and
  // class vectors are read into registers through global-address loads
  float xfr[FC > 0 ? FC : 1], xsr[KC > 0 ? KC : 1];
  if (FC > 0 && P.src_feat) {
#pragma unroll
    for (int f = 0; f < (FC > 0 ? FC : 1); ++f) xfr[f] = ld_global(P.src_feat + (size_t)r * F + f);
  }
  if (KC > 0 && P.src_sem) {
#pragma unroll
    for (int k = 0; k < (KC > 0 ? KC : 1); ++k) xsr[k] = ld_global(P.src_sem + (size_t)r * KS + k);
  }
  const float* xf = P.src_feat ? (FC > 0 ? xfr : P.src_feat + (size_t)r * kc.F) : nullptr;
  const float* xs = P.src_sem ? (KC > 0 ? xsr : P.src_sem + (size_t)r * kc.Ks) : nullptr;
  float xg[2] = {0.0f, 0.0f};
  if (kc.use_gtype) {
    xg[0] = ld_global(P.src_geo + 2 * (size_t)r);
    xg[1] = ld_global(P.src_geo + 2 * (size_t)r + 1);
  }
  float q0, q1, q2;
  affine3(mp.Rq, mp.Tq, x0, x1, x2, q0, q1, q2);
  const float rq = sqrtf(d2t) * 1.001f + 1e-4f * (1.0f + fmaxf(fabsf(q0), fmaxf(fabsf(q1), fabsf(q2))));
  const CellBox B = cell_box(GL, q0, q1, q2, rq);
  // a passing target's key is its index; ~0 for the others
  auto eval = [&](uint32_t pidx, float4& y4, float& y0, float& y1, float& y2, float& a) -> uint64_t {
    y4 = ld_global(GL.pos + pidx);
    float yfr[FC > 0 ? FC : 1], ysr[KC > 0 ? KC : 1];
    if (FC > 0) {
#pragma unroll
      for (int f = 0; f < (FC > 0 ? FC : 1); ++f) yfr[f] = ld_global(GL.feat + (size_t)pidx * F + f);
    }
    if (KC > 0) {
#pragma unroll
      for (int k = 0; k < (KC > 0 ? KC : 1); ++k) ysr[k] = ld_global(GL.sem + (size_t)pidx * KS + k);
    }
    affine3(mp.A, mp.b, y4.x, y4.y, y4.z, y0, y1, y2);
    const bool pass = pair_kernel<FC, KC>(kc, ek, x0, x1, x2, y0, y1, y2, d2t, qg, l, xf,
                                          FC > 0 ? yfr : (FC != 0 ? GL.feat + (size_t)pidx * F : nullptr), xs,
                                          KC > 0 ? ysr : (KC != 0 ? GL.sem + (size_t)pidx * KS : nullptr), xg,
                                          kc.use_gtype ? GL.geo + 2 * (size_t)pidx : nullptr, a);
    return pass ? (uint64_t)__float_as_uint(y4.w) : ~0ull;
  };
  uint64_t thr;
  int tsh;
  select_smallest<64>(
      [&](auto&& fn) { for_each_in_box<64>(GL, B, g, fn); }, g, K, hist,
      [&](uint32_t pidx) {
        float4 y4;
        float y0, y1, y2, a;
        return eval(pidx, y4, y0, y1, y2, a);
      },
      thr, tsh);
  uint32_t stored = 0;
  for_each_in_box<64>(GL, B, g, [&](bool valid, uint32_t pidx) {
    bool take = false;
    float a = 0.0f, y0 = 0.0f, y1 = 0.0f, y2 = 0.0f;
    float4 y4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid) {
      const uint64_t key = eval(pidx, y4, y0, y1, y2, a);
      take = selected(key, thr, tsh);
    }
    const uint64_t m = __ballot(take);
    const uint32_t slot = stored + (uint32_t)__popcll(m & ((g == 0) ? 0ull : (~0ull >> (64 - g))));
    if (take && slot < K) {
      store_pair(P, mode, r, K, slot, pidx, y4, a);
      if (mode == MODE_ALIGN) {
        const float c0 = x1 * y2 - x2 * y1, c1 = x2 * y0 - x0 * y2, c2 = x0 * y1 - x1 * y0;
        acc[0] += (double)(c0 * a);
        acc[1] += (double)(c1 * a);
        acc[2] += (double)(c2 * a);
        acc[3] += (double)((y0 - x0) * a);
        acc[4] += (double)((y1 - x1) * a);
        acc[5] += (double)((y2 - x2) * a);
      }
      acc[6] += (double)(kc.ip_ad2 ? sq_dist(x0, x1, x2, y0, y1, y2) * a : a);
    }
    stored += (uint32_t)__popcll(m);
  });
  return min(stored, K);
}

// ---------------------------------------------------------------------------
// Step terms (compute_step_size_xi + compute_step_size_poly_coeff, CvoGPU.cu:
// 333-462): block partials part_s[block] = B, C, D, E (FP64).
// ---------------------------------------------------------------------------

__device__ __forceinline__ void cross_f(float a0, float a1, float a2, float b0, float b1, float b2, float& o0,
                                        float& o1, float& o2) {
  o0 = a1 * b2 - a2 * b1;
  o1 = a2 * b0 - a0 * b2;
  o2 = a0 * b1 - a1 * b0;
}

// The pass's flow, omega / c and v / d (compute_flow_gpu_no_eigen,
// CvoGPU.cu:2057-2060).
__device__ __forceinline__ void scaled_flow(const ProblemState* st, const KConsts& kc, double tot[6]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    tot[c] = st->flow[c] / (double)kc.c;
    tot[3 + c] = st->flow[3 + c] / (double)kc.d;
  }
}

// The flow's direction as the step terms use it, in float: normalised
// (compute_flow, CvoGPU.cu:2099-2104), or as summed in the adaptive-lengthscale
// loop (AdaptiveCvoGPU.cu:839-840).
struct StepDir {
  float w0, w1, w2, v0, v1, v2;
};
__device__ __forceinline__ StepDir step_direction(const KConsts& kc, const double tot[6]) {
  double n2 = 0.0;
#pragma unroll
  for (int c = 0; c < 6; ++c) n2 += tot[c] * tot[c];
  const double nrm = (n2 > 0.0 && !kc.adaptive) ? sqrt(n2) : 1.0;
  StepDir d;
  d.w0 = (float)(tot[0] / nrm); d.w1 = (float)(tot[1] / nrm); d.w2 = (float)(tot[2] / nrm);
  d.v0 = (float)(tot[3] / nrm); d.v1 = (float)(tot[4] / nrm); d.v2 = (float)(tot[5] / nrm);
  return d;
}

// Step terms of one row's pairs l, l + L, ... (row: its cnt stored pairs),
// added to acc in that order.
constexpr int kStepLoads = 4;  // pairs whose loads are in flight together per thread
__device__ __forceinline__ void step_row(const KConsts& kc, const GridLevel& G, const Maps& mp, const StepDir& dir,
                                         const float4& x4, float ell, const uint2* row, uint32_t cnt, uint32_t l,
                                         uint32_t L, double acc[4]) {
  const float w0 = dir.w0, w1 = dir.w1, w2 = dir.w2, v0 = dir.v0, v1 = dir.v1, v2 = dir.v2;
  float x0 = x4.x, x1 = x4.y, x2 = x4.z;
  if (mp.src_xf) {
    float t0, t1, t2;
    affine3(mp.As, mp.bs, x0, x1, x2, t0, t1, t2);
    x0 = t0; x1 = t1; x2 = t2;
  }
  float temp_ell = ell;
  if (kc.range_ell_in_step) {
    const float px = sqrtf(x0 * x0 + x1 * x1 + x2 * x2);
    temp_ell = (float)(((double)px / 500.0 + 1.0) * (double)ell);
  }
  const float tc = (float)(1.0 / (2.0 * (double)temp_ell * (double)temp_ell));
  // one pair's Taylor terms, summed into acc in pair order
  auto step_pair = [&](const float a, const float4 y4) {
    float z0, z1, z2;
    affine3(mp.A, mp.b, y4.x, y4.y, y4.z, z0, z1, z2);
    // xi^k z: xiz = w x z + v, xi^{k+1} z = w x xi^k z
    float a0, a1, a2, b0, b1, b2, c0, c1, c2, d0, d1, d2;
    cross_f(w0, w1, w2, z0, z1, z2, a0, a1, a2);
    a0 += v0; a1 += v1; a2 += v2;
    cross_f(w0, w1, w2, a0, a1, a2, b0, b1, b2);
    cross_f(w0, w1, w2, b0, b1, b2, c0, c1, c2);
    cross_f(w0, w1, w2, c0, c1, c2, d0, d1, d2);
    const float df0 = x0 - z0, df1 = x1 - z1, df2 = x2 - z2;
    const float normxiz2 = a0 * a0 + a1 * a1 + a2 * a2;
    const float xiz_dot_xi2z = -(a0 * b0 + a1 * b1 + a2 * b2);
    const float epsil_const = (b0 * b0 + b1 * b1 + b2 * b2) + 2.0f * (a0 * c0 + a1 * c1 + a2 * c2);
    const float beta = (float)(-2.0 * (double)tc * (double)(a0 * df0 + a1 * df1 + a2 * df2));
    const float gamma = -tc * (normxiz2 + 2.0f * (b0 * df0 + b1 * df1 + b2 * df2));
    const float delta = (float)(2.0 * (double)tc * (double)(xiz_dot_xi2z - (c0 * df0 + c1 * df1 + c2 * df2)));
    const float epsil = -tc * (epsil_const + 2.0f * (d0 * df0 + d1 * df1 + d2 * df2));
    const double ad = (double)a, bd = (double)beta, gd = (double)gamma;
    acc[0] += (double)(a * beta);
    acc[1] += ad * (gd + (double)(beta * beta) / 2.0);
    acc[2] += ad * ((double)(delta + beta * gamma) + (double)(beta * beta * beta) / 6.0);
    acc[3] += ad * ((double)(epsil + beta * delta) + 0.5 * bd * bd * gd + 0.5 * gd * gd +
                    (1.0 / 24.0) * bd * bd * bd * bd);
  };
  // kStepLoads pairs a trip: their slots, then their target gathers, go out
  // before the first pair is summed
  uint32_t s = l;
  for (; s + (kStepLoads - 1) * L < cnt; s += kStepLoads * L) {
    uint2 e[kStepLoads];
    float4 y[kStepLoads];
#pragma unroll
    for (int u = 0; u < kStepLoads; ++u) e[u] = ld_global(row + s + u * L);
#pragma unroll
    for (int u = 0; u < kStepLoads; ++u) y[u] = ld_global(G.pos + e[u].x);
#pragma unroll
    for (int u = 0; u < kStepLoads; ++u) step_pair(__uint_as_float(e[u].y), y[u]);
  }
  for (; s < cnt; s += L) {
    const uint2 e = ld_global(row + s);
    step_pair(__uint_as_float(e.y), ld_global(G.pos + e.x));
  }
}

// Lanes per row of a problem's next pass (4, 8 or 16).
__device__ __forceinline__ int state_group(const ProblemState* st) {
  return st->group == 4 ? 4 : (st->group == 8 ? 8 : 16);
}

}  // namespace cvo
