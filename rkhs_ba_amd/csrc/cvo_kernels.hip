// gfx950 kernels of the CVO two-view loop.
//
//   grid_cell_count / grid_gather : uniform-grid levels over a target cloud
//   src_sort_keys / src_gather    : spatially sorted copy of the source rows
//   assoc_kernel                  : ell-ball search + product kernel + row store
//                                   (first K by target index) + fused flow
//                                   (fill_in_A_mat_gpu CvoGPU.cu:951-1099 and
//                                   compute_flow_gpu_no_eigen :2001-2062)
//   overflow_kernel               : the pass totals, plus the rows whose
//                                   passing pairs exceed the cap K (their K
//                                   smallest passing target indices)
//   step_kernel                   : Taylor step terms (:333-462); its last
//                                   block runs the device controller
//                                   (:464-544, :1289-1433)
//
// Rows are processed by groups of G = 4, 8 or 16 lanes (256 / G rows per
// 256-thread block), G chosen per iteration from the lengthscale.  Reductions
// are block partials summed in fixed order, so results are bitwise
// reproducible run to run.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "cvo_internal.h"
#include "cvo_device.h"
#include "cvo_assoc.h"
#include "cvo_ball.h"
#include "cvo_controller.h"

namespace cvo {

// ---------------------------------------------------------------------------
// Grid construction
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint32_t cell_of(float x, float y, float z, float ox, float oy, float oz, float inv_h,
                                            int nx, int ny, int nz) {
  int cx = (int)floorf((x - ox) * inv_h);
  int cy = (int)floorf((y - oy) * inv_h);
  int cz = (int)floorf((z - oz) * inv_h);
  cx = min(max(cx, 0), nx - 1);
  cy = min(max(cy, 0), ny - 1);
  cz = min(max(cz, 0), nz - 1);
  return ((uint32_t)cz * (uint32_t)ny + (uint32_t)cy) * (uint32_t)nx + (uint32_t)cx;
}

__global__ void grid_cell_count(const float* __restrict__ xyz, int n, float ox, float oy, float oz, float inv_h,
                                int nx, int ny, int nz, uint32_t* __restrict__ key, uint32_t* __restrict__ count) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const uint32_t c = cell_of(xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2], ox, oy, oz, inv_h, nx, ny, nz);
  key[j] = c;
  atomicAdd(&count[c], 1u);
}

// Zero fill, in place of a memset node (which a caller's graph capture
// should not record).
__global__ void zero_u32(uint32_t* __restrict__ v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) v[i] = 0u;
}

__global__ void iota_u32(uint32_t* __restrict__ v, int n) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) v[j] = (uint32_t)j;
}

// The attributes of point j to sorted place s.
__device__ __forceinline__ void gather_attributes(int s, uint32_t j, const float* feat, int F, const float* sem, int K,
                                                  const float* geo, float* feat_s, float* sem_s, float* geo_s) {
  if (feat_s)
    for (int f = 0; f < F; ++f) feat_s[(size_t)s * F + f] = feat[(size_t)j * F + f];
  if (sem_s)
    for (int k = 0; k < K; ++k) sem_s[(size_t)s * K + k] = sem[(size_t)j * K + k];
  if (geo_s) {
    geo_s[2 * (size_t)s] = geo[2 * (size_t)j];
    geo_s[2 * (size_t)s + 1] = geo[2 * (size_t)j + 1];
  }
}

// Gathers the cloud into sorted order: pos = (x, y, z, original id bits).
__global__ void gather_sorted(const uint32_t* __restrict__ order, int n, const float* __restrict__ xyz,
                              const float* __restrict__ feat, int F, const float* __restrict__ sem, int K,
                              const float* __restrict__ geo, float4* __restrict__ pos, float* __restrict__ feat_s,
                              float* __restrict__ sem_s, float* __restrict__ geo_s, uint32_t* __restrict__ inv_perm) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint32_t j = order[s];
  pos[s] = make_float4(xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2], __uint_as_float(j));
  gather_attributes(s, j, feat, F, sem, K, geo, feat_s, sem_s, geo_s);
  if (inv_perm) inv_perm[j] = (uint32_t)s;
}

// 30-bit Morton key of a point in its cloud's bounding box (source row order).
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

struct MortonBox {
  float o[3], s[3];  // a coordinate x becomes (x - o) s
};
__device__ __forceinline__ uint32_t morton_of(const MortonBox& B, float x, float y, float z) {
  uint32_t a = (uint32_t)fminf(fmaxf((x - B.o[0]) * B.s[0], 0.0f), 1023.0f);
  uint32_t b = (uint32_t)fminf(fmaxf((y - B.o[1]) * B.s[1], 0.0f), 1023.0f);
  uint32_t c = (uint32_t)fminf(fmaxf((z - B.o[2]) * B.s[2], 0.0f), 1023.0f);
  return spread10(a) | (spread10(b) << 1) | (spread10(c) << 2);
}

__global__ void morton_keys(const float* __restrict__ xyz, int n, MortonBox B, uint32_t* __restrict__ key) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) key[j] = morton_of(B, xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2]);
}

// Small clouds (sorts_in_a_block): all levels of a grid in two launches (and the
// source rows in one or two) instead of six to ten launches a level, each of
// which lasts longer than its work.  One block a level sorts (key, index) words
// in LDS, bitonic, two strides a trip; unique words, so the order is the stable
// one of the general path.  Latency-bound: 49 trips with a barrier each at 8192
// words.  The set-up of a registration with ten levels 404 -> 176 us at 2000
// points, 518 -> 308 at 8192.
__device__ __forceinline__ void order_words(uint64_t& a, uint64_t& b, bool up) {
  const uint64_t lo = a < b ? a : b, hi = a < b ? b : a;
  a = up ? lo : hi;
  b = up ? hi : lo;
}
template <class Key>
__device__ __forceinline__ void small_sort(const float* xyz, int n, int padded, Key key, float4* pos,
                                           uint32_t* inv_perm) {
  extern __shared__ uint64_t s_word[];
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int j = tid; j < padded; j += nt)
    s_word[j] = j < n ? (uint64_t)key(xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2]) << 32 | (uint32_t)j : ~0ull;
  __syncthreads();
  for (int k = 2; k <= padded; k <<= 1) {
    int j = k >> 1;
    for (; j >= 2; j >>= 2) {
      const int h = j >> 1;
      for (int t = tid; t < padded / 4; t += nt) {
        const int i = (t & ~(h - 1)) * 4 + (t & (h - 1));
        const bool up = (i & k) == 0;
        uint64_t a = s_word[i], b = s_word[i + h], c = s_word[i + 2 * h], d = s_word[i + 3 * h];
        order_words(a, c, up);
        order_words(b, d, up);
        order_words(a, b, up);
        order_words(c, d, up);
        s_word[i] = a;
        s_word[i + h] = b;
        s_word[i + 2 * h] = c;
        s_word[i + 3 * h] = d;
      }
      __syncthreads();
    }
    if (j == 1) {
      for (int t = tid; t < padded / 2; t += nt) {
        const bool up = (2 * t & k) == 0;
        uint64_t a = s_word[2 * t], b = s_word[2 * t + 1];
        order_words(a, b, up);
        s_word[2 * t] = a;
        s_word[2 * t + 1] = b;
      }
      __syncthreads();
    }
  }
  for (int s = tid; s < n; s += nt) {
    const uint32_t j = (uint32_t)s_word[s];
    pos[s] = make_float4(xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2], __uint_as_float(j));
    if (inv_perm) inv_perm[j] = (uint32_t)s;
  }
}

__global__ __launch_bounds__(1024) void small_source_kernel(const float* __restrict__ xyz, int n, int padded,
                                                            MortonBox B, float4* __restrict__ pos) {
  small_sort(xyz, n, padded, [&](float x, float y, float z) { return morton_of(B, x, y, z); }, pos, nullptr);
}

// Block l: level l of G.
__global__ __launch_bounds__(1024) void small_levels_kernel(const float* __restrict__ xyz, int n, int padded, GridDev G) {
  const GridLevel L = G.lv[blockIdx.x];
  small_sort(xyz, n, padded, [&](float x, float y, float z) {
    return cell_of(x, y, z, L.ox, L.oy, L.oz, L.inv_h, L.nx, L.ny, L.nz);
  }, const_cast<float4*>(L.pos), const_cast<uint32_t*>(L.inv_perm));
}

__global__ void small_attributes_kernel(int n, const float4* __restrict__ pos, const float* __restrict__ feat, int F,
                                        const float* __restrict__ sem, int K, const float* __restrict__ geo,
                                        float* __restrict__ feat_s, float* __restrict__ sem_s,
                                        float* __restrict__ geo_s) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) gather_attributes(s, __float_as_uint(pos[s].w), feat, F, sem, K, geo, feat_s, sem_s, geo_s);
}

// Row y: level y; its first point_blocks blocks gather the attributes, each of the
// others fills kCellsPerBlock cell starts (cell c: the points before c's first)
// from the keys of the sorted points in that range of cells, which the positions
// give again.
constexpr int kCellsPerThread = 8, kCellsPerBlock = 256 * kCellsPerThread;
__global__ __launch_bounds__(256) void small_cells_kernel(int n, int point_blocks, GridDev G,
                                                          const float* __restrict__ feat, int F,
                                                          const float* __restrict__ sem, int K,
                                                          const float* __restrict__ geo) {
  const GridLevel L = G.lv[blockIdx.y];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < point_blocks) {
    const int s = blockIdx.x * 256 + tid;
    if (s < n)
      gather_attributes(s, __float_as_uint(L.pos[s].w), feat, F, sem, K, geo, const_cast<float*>(L.feat),
                        const_cast<float*>(L.sem), const_cast<float*>(L.geo));
    return;
  }
  const uint32_t entries = (uint32_t)L.nx * (uint32_t)L.ny * (uint32_t)L.nz + 1u;
  const uint32_t c0 = (blockIdx.x - (uint32_t)point_blocks) * kCellsPerBlock;
  if (c0 >= entries) return;
  const uint32_t c1 = c0 + kCellsPerBlock;
  auto key = [&](int s) {
    const float4 p = L.pos[s];
    return cell_of(p.x, p.y, p.z, L.ox, L.oy, L.oz, L.inv_h, L.nx, L.ny, L.nz);
  };
  auto first = [&](uint32_t c) {  // the first sorted point in cell c or later
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (key(mid) < c) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  __shared__ int s_first[kCellsPerBlock];
  __shared__ int s_min[256];
  const int lo = first(c0), hi = first(c1);
  for (int c = tid; c < kCellsPerBlock; c += 256) s_first[c] = hi;
  __syncthreads();
  for (int s = lo + tid; s < hi; s += 256) atomicMin(&s_first[key(s) - c0], s);
  __syncthreads();
  // minimum over the cells from c on
  int own[kCellsPerThread], m = hi;
#pragma unroll
  for (int u = kCellsPerThread - 1; u >= 0; --u) {
    m = min(m, s_first[tid * kCellsPerThread + u]);
    own[u] = m;
  }
  s_min[tid] = m;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int x = tid + o < 256 ? s_min[tid + o] : hi;
    __syncthreads();
    s_min[tid] = min(s_min[tid], x);
    __syncthreads();
  }
  const int rest = tid + 1 < 256 ? s_min[tid + 1] : hi;
  uint32_t* out = const_cast<uint32_t*>(L.cell_start);
#pragma unroll
  for (int u = 0; u < kCellsPerThread; ++u) {
    const uint32_t c = c0 + (uint32_t)(tid * kCellsPerThread + u);
    if (c < entries) out[c] = (uint32_t)min(own[u], rest);
  }
}

// Block partials of the association pass: part_a[block] = flow6, ip, -;
// part_cnt[block] = stored pairs, max row; summed into the problem state by
// the capped-row kernel that follows.

// LDS of one association block, sized for the most rows a block of the
// variant can hold (ROWS: 64 with the four-lane path, else 32; the K-nearest
// variant's histograms leave no room for more).
template <int FC, int KC, int ROWS>
struct AssocLds {
  static constexpr int FL = FC > 0 ? FC : (FC == 0 ? 1 : 64);
  static constexpr int KL = KC > 0 ? KC : (KC == 0 ? 1 : 64);
  static constexpr int kRows = ROWS;
  double row[ROWS][8];
  uint32_t cnt[ROWS];
  float feat[ROWS * FL];  // the block's source rows' features
  float sem[ROWS * KL];   // and class vectors
};

// Logical block lb of a problem with G lanes per row (256 / G rows); KNN:
// the K-nearest rows (hist: 256 bins per row).
template <int FC, int KC, int G, bool KNN, int ROWS>
__device__ __forceinline__ void assoc_block(const AssocProblem& P, const KConsts& kc, int lb,
                                            AssocLds<FC, KC, ROWS>& L, uint32_t* hist) {
  constexpr int RB = rows_per_block(G);
  static_assert(RB <= ROWS, "the block's rows exceed its LDS");
  const ProblemState* st = P.st;
  const int tid = threadIdx.x;
  const int g = tid & (G - 1);
  const int grp = tid / G;
  const int r = lb * RB + grp;
  const int mode = kc.mode;
  const float ell = st->ell;
  const int K = st->K;
  const int iter = st->iter;
  Maps mp;
  load_maps(st, mp);
  const ExactK ek = exact_consts(kc);
  // a copy: the pair stores below cannot alias it, so its fields stay in
  // registers instead of being reloaded after every store
  GridLevel GL = P.grid->lv[st->level];
  if constexpr (!KNN && ROWS != kMaxRowsPerBlock) {
    // batched launches have no vector registers to spare for what is the same
    // in all lanes
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      mp.A[i] = uni(mp.A[i]);
      mp.Rq[i] = uni(mp.Rq[i]);
      mp.As[i] = uni(mp.As[i]);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      mp.b[i] = uni(mp.b[i]);
      mp.Tq[i] = uni(mp.Tq[i]);
      mp.bs[i] = uni(mp.bs[i]);
    }
    GL = uniform_level(GL);
  }
  const int row0 = lb * RB;
  const int nrows = min(RB, P.n_src - row0);
  if (FC != 0) {
    const int F = Dim<FC>::get(kc.F);
    for (int t = tid; t < nrows * F; t += kBlock) L.feat[t] = ld_global(P.src_feat + (size_t)row0 * F + t);
  }
  if (KC != 0) {
    const int KS = Dim<KC>::get(kc.Ks);
    for (int t = tid; t < nrows * KS; t += kBlock) L.sem[t] = ld_global(P.src_sem + (size_t)row0 * KS + t);
  }
  __syncthreads();
  RowResult res;
#pragma unroll
  for (int c = 0; c < 7; ++c) res.acc[c] = 0.0;
  res.stored = 0;
  res.overflow = false;
  if (r < P.n_src) {
    if constexpr (KNN)
      knn_row<FC, KC, G>(P, kc, ek, GL, mp, r, g, mode, ell, K, ld_global(P.src_pos + r), L.feat + grp * Dim<FC>::get(kc.F),
                         L.sem + grp * Dim<KC>::get(kc.Ks), hist + grp * 256, res);
    else
      assoc_row<FC, KC, G, (ROWS == kMaxRowsPerBlock)>(P, kc, ek, GL, mp, r, g, mode, ell, K,
                                                       ld_global(P.src_pos + r),
                                                       L.feat + grp * Dim<FC>::get(kc.F),
                                                       L.sem + grp * Dim<KC>::get(kc.Ks), res);
  }
#pragma unroll
  for (int c = 0; c < 7; ++c) {
    double v = res.acc[c];
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, G);
    res.acc[c] = v;
  }
  if (g == 0) {
    uint32_t cnt = 0;
    if (r < P.n_src) {
      // a capped row is counted by the capped-row kernel, which rewrites it
      cnt = res.overflow ? 0u : res.stored;
      st_global(P.counts + r, cnt);
      if (res.overflow) {
        st_global(P.ovf_stamp + r, (uint32_t)iter + 1u);
        atomicAdd(&P.st->n_overflow, 1u);
      }
    }
#pragma unroll
    for (int c = 0; c < 7; ++c) L.row[grp][c] = res.overflow ? 0.0 : res.acc[c];
    L.cnt[grp] = cnt;
  }
  __syncthreads();
  if (tid < 7) {
    double s = 0.0;
    for (int q = 0; q < RB; ++q) s += L.row[q][tid];
    st_global(P.part_a + (size_t)lb * 8 + tid, s);
  } else if (tid == 7) {
    uint32_t nz = 0, mx = 0;
    for (int q = 0; q < RB; ++q) {
      nz += L.cnt[q];
      mx = max(mx, L.cnt[q]);
    }
    st_global(P.part_cnt + (size_t)lb * 2, nz);
    st_global(P.part_cnt + (size_t)lb * 2 + 1, mx);
  }
}

// Fixed-order tree over red[c][0..W): sums, except the max-row column 8.
// Every thread of the block takes part; red[c][0] holds the result.
template <int W>
__device__ __forceinline__ void tree10(double (*red)[W]) {
  const int tid = threadIdx.x;
  for (int w = W / 2; w > 0; w >>= 1) {
    __syncthreads();
    for (int t = tid; t < 10 * w; t += kBlock) {
      const int c = t / w, i = t - c * w;
      red[c][i] = (c == 8) ? fmax(red[c][i], red[c][i + w]) : red[c][i] + red[c][i + w];
    }
  }
  __syncthreads();
}

// Active association blocks of a problem at a lane count.
__device__ __forceinline__ int active_blocks(const AssocProblem& P, int group) {
  const int rb = kBlock / group;
  return (P.n_src + rb - 1) / rb;
}

// One launch covers every problem; a problem owns P.n_blocks blocks (its rows
// at the largest lane count) and uses a prefix of them at its current lane
// count.  With xcd_remap the active blocks are renumbered so that each
// XCD holds one contiguous range of rows.
// Register budget: see assoc_kernel.
// FOUR: the four-lanes-per-row path is compiled in (single-problem kernels
// only: it raises the batched variant's register count past its budget; the
// host never selects four lanes for a batched launch).
template <int FC, int KC, bool KNN, bool FOUR>
__device__ __forceinline__ void assoc_pass(const AssocProblem& P, const KConsts& kc) {
  const ProblemState* st = P.st;
  if (st->done) return;
  const int group = state_group(st);
  const int n_act = active_blocks(P, group);
  int lb = (int)blockIdx.x - P.block_begin;
  if (lb >= n_act) return;  // uniform
  if (kc.xcd_remap) lb = xcd_block(lb, n_act);
  __shared__ AssocLds<FC, KC, FOUR ? kMaxRowsPerBlock : kKnnRowsPerBlock> L;
  if constexpr (KNN) {
    __shared__ uint32_t hist[kKnnRowsPerBlock * 256];
    switch (group) {
      case 8: assoc_block<FC, KC, 8, true>(P, kc, lb, L, hist); break;
      default: assoc_block<FC, KC, 16, true>(P, kc, lb, L, hist); break;
    }
  } else {
    switch (group) {
      // two lane counts keep the kernel within its register budget
      case 4:
        if constexpr (FOUR) assoc_block<FC, KC, 4, false>(P, kc, lb, L, nullptr);
        break;
      case 8: assoc_block<FC, KC, 8, false>(P, kc, lb, L, nullptr); break;
      default: assoc_block<FC, KC, 16, false>(P, kc, lb, L, nullptr); break;
    }
  }
}

// ONE: a single problem, its descriptor by value in the kernel arguments (read
// with scalar loads, no dependent load before the first state read).
// Occupancy: five waves per SIMD for one problem (96 VGPRs; six spill 96 bytes: the
// 60k street registration 125 against 157 ms).  Batched launches hold the maps and
// the grid level in scalar registers and run at four (106 VGPRs, none spilled):
// 96 starts over 20k points, 1000 iterations, 16 lanes above ell 0.158 and 8 below
// 1.58 s, untuned 1.54; at five waves 31 registers spill, 1.71 and 1.74 (40
// iterations at ell 0.5 8 % faster, at 0.08 14 % slower); with the maps in vector
// registers at four 1.61.
template <int FC, int KC, bool ONE>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(ONE ? 5 : 4))) void assoc_kernel(
    const AssocProblem* __restrict__ probs, int n_probs, KConsts kc, AssocProblem one) {
  if constexpr (ONE) {
    assoc_pass<FC, KC, false, true>(one, kc);
  } else {
    // a register copy of the problem: the pair stores cannot alias it
    const AssocProblem P = probs[find_problem(probs, n_probs, (int)blockIdx.x)];
    assoc_pass<FC, KC, false, false>(P, kc);
  }
}

// The K-nearest association pass (is_using_kdtree), same launch shape and
// outputs; rows never exceed their cap, so no capped-row work follows.
template <int FC, int KC, bool ONE>
__global__ __launch_bounds__(kBlock) void knn_assoc_kernel(const AssocProblem* __restrict__ probs, int n_probs,
                                                           KConsts kc, AssocProblem one) {
  if constexpr (ONE) {
    assoc_pass<FC, KC, true, false>(one, kc);
  } else {
    const AssocProblem P = probs[find_problem(probs, n_probs, (int)blockIdx.x)];
    assoc_pass<FC, KC, true, false>(P, kc);
  }
}

// ---------------------------------------------------------------------------
// Totals of an association pass, and the rows whose passing pairs exceed the
// cap, which keep their first K passing targets by index (the reference's
// scan over all targets in ascending index, CvoGPU.cu:994-996).  Each block sums a slice of the
// association block partials, adds its capped rows and publishes
// part_ovf[block] = flow6, ip, stored, max row; the last block writes the
// problem's totals (raw flow sums, ip, stored pairs, longest row).
// ---------------------------------------------------------------------------

// The pass totals of a problem by one block: thread t takes association
// blocks t, t + 256, ... (four at a time, for loads in flight), then a fixed
// tree: wave shuffles, then the four waves in order.
__device__ __forceinline__ void pass_totals_one_block(const AssocProblem& P, ProblemState* st) {
  const int tid = threadIdx.x;
  const int n_act = active_blocks(P, state_group(st));
  double acc[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  double nz = 0.0, mx = 0.0;
#pragma unroll 4
  for (int b = tid; b < n_act; b += kBlock) {
    const double2* pa = reinterpret_cast<const double2*>(P.part_a + (size_t)b * 8);
    const double2 q0 = pa[0], q1 = pa[1], q2 = pa[2], q3 = pa[3];
    const uint2 cn = reinterpret_cast<const uint2*>(P.part_cnt)[b];
    acc[0] += q0.x; acc[1] += q0.y; acc[2] += q1.x; acc[3] += q1.y;
    acc[4] += q2.x; acc[5] += q2.y; acc[6] += q3.x;
    nz += (double)cn.x;
    mx = fmax(mx, (double)cn.y);
  }
  __shared__ double s_w[9][kBlock / 64];
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    double v = c < 7 ? acc[c] : (c == 7 ? nz : mx);
    for (int o = 32; o > 0; o >>= 1) {
      const double u = __shfl_xor(v, o, 64);
      v = c == 8 ? fmax(v, u) : v + u;
    }
    if (lane == 0) s_w[c][wave] = v;
  }
  __syncthreads();
  if (tid == 0) {
    double t[9];
    for (int c = 0; c < 9; ++c) {
      t[c] = 0.0;
      for (int w = 0; w < kBlock / 64; ++w) t[c] = c == 8 ? fmax(t[c], s_w[c][w]) : t[c] + s_w[c][w];
    }
    for (int c = 0; c < 6; ++c) st->flow[c] = t[c];
    st->ip = t[6];
    st->nnz = (uint64_t)t[7];
    st->max_row = (uint32_t)t[8];
    st->level_assoc = st->level;
  }
}


template <int FC, int KC>
__device__ __forceinline__ void overflow_body(const AssocProblem& P, const KConsts& kc) {
  ProblemState* st = P.st;
  if (st->done) return;
  const int tid = threadIdx.x;
  const int mode = kc.mode;
  if (st->n_overflow == 0) {
    // no capped row: block 0 alone sums every association partial (no
    // cross-block publication), the other blocks have nothing to do
    if (blockIdx.x == 0) pass_totals_one_block(P, st);
    return;  // uniform per block
  }
  // (a) this block's slice of the association block partials, in fixed order
  __shared__ double s_tot[10][128];
  {
    const int n_act = active_blocks(P, state_group(st));
    const int per = (n_act + kOvfBlocks - 1) / kOvfBlocks;
    const int b0 = blockIdx.x * per, b1 = min(n_act, b0 + per);
    for (int t = tid; t < 10 * 128; t += kBlock) {
      const int c = t / 128, i = t - c * 128;
      double v = 0.0;
      for (int b = b0 + i; b < b1; b += 128) {
        if (c < 7) v += ld_global(P.part_a + (size_t)b * 8 + c);
        else if (c == 7) v += (double)ld_global(P.part_cnt + (size_t)b * 2);
        else if (c == 8) v = fmax(v, (double)ld_global(P.part_cnt + (size_t)b * 2 + 1));
      }
      s_tot[c][i] = v;
    }
    tree10<128>(s_tot);
  }
  double blk_acc[7];
#pragma unroll
  for (int c = 0; c < 7; ++c) blk_acc[c] = s_tot[c][0];
  uint32_t blk_nnz = (uint32_t)s_tot[7][0], blk_max = (uint32_t)s_tot[8][0];
  __syncthreads();
  // (b) rows whose passing pairs exceed the cap (uniform branch)
  if (st->n_overflow != 0) {
  const float ell = st->ell;
  const uint32_t K = (uint32_t)st->K;
  const uint32_t stamp = (uint32_t)st->iter + 1u;
  Maps mp;
  load_maps(st, mp);
  const ExactK ek = exact_consts(kc);
  const GridLevel G = P.grid->lv[st->level];  // a register copy, as in the association
  const int F = Dim<FC>::get(kc.F);
  const int KS = Dim<KC>::get(kc.Ks);
  const int chunk = (P.n_src + kOvfBlocks - 1) / kOvfBlocks;
  const int r0 = blockIdx.x * chunk, r1 = min(P.n_src, r0 + chunk);
  __shared__ uint32_t s_wave[kBlock / 64];
  __shared__ double s_red[kBlock];
  if (kc.use_geo) {
    // the chunk's capped rows, one wave per row in turn (wave w takes the
    // w-th, (w+4)-th, ... capped row of the chunk)
    __shared__ uint32_t s_hist[kBlock / 64][256];
    __shared__ double s_wacc[kBlock / 64][9];
    const int lane = tid & 63, wave = tid >> 6;
    double wacc[7] = {0, 0, 0, 0, 0, 0, 0};
    uint32_t wnnz = 0, wmax = 0, seen = 0;
    for (int base = r0; base < r1; base += 64) {
      const int rr = base + lane;
      uint64_t m = __ballot(rr < r1 && ld_global(P.ovf_stamp + rr) == stamp);
      while (m) {
        const int b = __ffsll((unsigned long long)m) - 1;
        m &= m - 1;
        if ((int)(seen % (kBlock / 64)) == wave) {
          const int r = base + b;
          double racc[7] = {0, 0, 0, 0, 0, 0, 0};
          const uint32_t kept = capped_row_ball<FC, KC>(P, kc, ek, G, mp, r, ell, K, s_hist[wave], racc, mode);
          if (lane == 0) st_global(P.counts + r, kept);
#pragma unroll
          for (int c = 0; c < 7; ++c) wacc[c] += racc[c];
          wnnz += kept;
          wmax = max(wmax, kept);
        }
        seen++;
      }
    }
#pragma unroll
    for (int c = 0; c < 7; ++c) {
      double v = wacc[c];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (lane == 0) s_wacc[wave][c] = v;
    }
    if (lane == 0) {
      s_wacc[wave][7] = (double)wnnz;
      s_wacc[wave][8] = (double)wmax;
    }
    __syncthreads();
    // every thread folds the waves in the same order (threads 0-7 publish)
    for (int w = 0; w < kBlock / 64; ++w) {
#pragma unroll
      for (int c = 0; c < 7; ++c) blk_acc[c] += s_wacc[w][c];
      blk_nnz += (uint32_t)s_wacc[w][7];
      blk_max = max(blk_max, (uint32_t)s_wacc[w][8]);
    }
  } else
  for (int r = r0; r < r1; ++r) {
    if (ld_global(P.ovf_stamp + r) != stamp) continue;  // uniform
    float4 x4 = ld_global(P.src_pos + r);
    float x0 = x4.x, x1 = x4.y, x2 = x4.z;
    if (mp.src_xf) {
      float t0, t1, t2;
      affine3(mp.As, mp.bs, x0, x1, x2, t0, t1, t2);
      x0 = t0; x1 = t1; x2 = t2;
    }
    const float l = kc.fixed_ell ? ell : range_ell(ell, x0, x1, x2);
    const float d2t = kc.use_geo ? (float)(-2.0 * (double)l * (double)l * (double)kc.lg) : 1.0f;
    const float qg = (float)(1.0 / (2.0 * (double)l * (double)l));
    const float* xf = P.src_feat ? P.src_feat + (size_t)r * kc.F : nullptr;
    const float* xs = P.src_sem ? P.src_sem + (size_t)r * kc.Ks : nullptr;
    float xg[2] = {0.0f, 0.0f};
    if (kc.use_gtype) {
      xg[0] = ld_global(P.src_geo + 2 * (size_t)r);
      xg[1] = ld_global(P.src_geo + 2 * (size_t)r + 1);
    }
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    uint32_t stored = 0;
    for (int base = 0; base < P.n_tgt && stored < K; base += kBlock) {
      const int j = base + tid;
      bool pass = false;
      float a = 0.0f, y0 = 0.0f, y1 = 0.0f, y2 = 0.0f;
      if (j < P.n_tgt) {
        affine3(mp.A, mp.b, ld_global(P.tgt_xyz + 3 * (size_t)j), ld_global(P.tgt_xyz + 3 * (size_t)j + 1), ld_global(P.tgt_xyz + 3 * (size_t)j + 2),
                y0, y1, y2);
        pass = pair_kernel<FC, KC>(kc, ek, x0, x1, x2, y0, y1, y2, d2t, qg, l, xf,
                                   FC != 0 ? P.tgt_feat + (size_t)j * F : nullptr, xs,
                                   KC != 0 ? P.tgt_sem + (size_t)j * KS : nullptr, xg,
                                   kc.use_gtype ? P.tgt_geo + 2 * (size_t)j : nullptr, a);
      }
      // block-wide exclusive prefix of pass flags, in index order
      const uint64_t m = __ballot(pass);
      const int lane = tid & 63, wave = tid >> 6;
      if (lane == 0) s_wave[wave] = (uint32_t)__popcll(m);
      __syncthreads();
      uint32_t before = 0, tot = 0;
      for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wave) before += s_wave[w];
        tot += s_wave[w];
      }
      before += (uint32_t)__popcll(m & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
      const uint32_t slot = stored + before;
      if (pass && slot < K) {
        const float4 y4 =
            make_float4(ld_global(P.tgt_xyz + 3 * (size_t)j), ld_global(P.tgt_xyz + 3 * (size_t)j + 1), ld_global(P.tgt_xyz + 3 * (size_t)j + 2), 0.0f);
        store_pair(P, mode, r, K, slot, G.inv_perm[j], y4, a);
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
      stored += tot;
      __syncthreads();
    }
    const uint32_t kept = min(stored, K);
    if (tid == 0) st_global(P.counts + r, kept);
    blk_nnz += kept;
    blk_max = max(blk_max, kept);
    for (int c = 0; c < 7; ++c) {
      s_red[tid] = acc[c];
      __syncthreads();
      for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (tid < w) s_red[tid] += s_red[tid + w];
        __syncthreads();
      }
      blk_acc[c] += s_red[0];
      __syncthreads();
    }
  }
  }
  // (c) the block's partial (its slice plus its capped rows); the last block
  // sums all blocks' partials in fixed order into the problem state
  double* out = P.part_ovf + (size_t)blockIdx.x * 10;
  __shared__ int s_last;
  if (tid < 64) {
    if (tid < 7) st_dev(&out[tid], blk_acc[tid]);
    if (tid == 7) {
      st_dev(&out[7], (double)blk_nnz);
      st_dev(&out[8], (double)blk_max);
      st_dev(&out[9], 0.0);
    }
    wait_stores();
    if (tid == 0) s_last = (count_in(&st->blocks_done_ovf) == (uint32_t)(gridDim.x - 1)) ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;  // uniform
  for (int t = tid; t < 10 * 128; t += kBlock) {
    const int c = t / 128, i = t - c * 128;
    s_tot[c][i] = (i < (int)gridDim.x) ? ld_dev(&P.part_ovf[(size_t)i * 10 + c]) : 0.0;
  }
  tree10<128>(s_tot);
  if (tid == 0) {
    for (int c = 0; c < 6; ++c) st->flow[c] = s_tot[c][0];
    st->ip = s_tot[6][0];
    st->nnz = (uint64_t)s_tot[7][0];
    st->max_row = (uint32_t)s_tot[8][0];
    st->level_assoc = st->level;
    st_dev(&st->blocks_done_ovf, 0u);
  }
}

// A single problem's descriptor comes by value in the kernel arguments (no
// dependent load before the first state read); several come from memory.
template <int FC, int KC, bool ONE>
__global__ __launch_bounds__(kBlock) void overflow_kernel(const AssocProblem* __restrict__ probs, KConsts kc,
                                                          AssocProblem one) {
  if constexpr (ONE) overflow_body<FC, KC>(one, kc);
  else {
    const AssocProblem P = probs[blockIdx.y];  // a register copy: stores cannot alias it
    overflow_body<FC, KC>(P, kc);
  }
}

// The self-association problems of an adaptive-lengthscale run after a step
// (adaptive_follow).  One thread.
__global__ void adaptive_sync_kernel(const AssocProblem* __restrict__ probs, KConsts kc) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const ProblemState* s0 = probs[0].st;
  for (int q = 1; q < 3; ++q) {
    const GridDev* grid = probs[q].grid;
    float h[kMaxLevels];
    for (int l = 0; l < kMaxLevels; ++l) h[l] = grid->lv[l].h;
    adaptive_follow(probs[q].st, s0, q, kc, h, grid->n_levels);
  }
}

// The controller step of a problem, run by the step pass's last block: step
// coefficients summed over the step blocks in fixed order, then the scalar
// controller on thread 0 with the state staged in LDS.
__device__ __forceinline__ void controller_tail(const AssocProblem& P, const KConsts& kc, const double tot[6], int nsb) {
  ProblemState* st = P.st;
  const int tid = threadIdx.x;
  __shared__ ProblemState s_st;
  __shared__ float s_h[kMaxLevels];
  __shared__ int s_nl;
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(st);
    uint32_t* dst = reinterpret_cast<uint32_t*>(&s_st);
    for (int i = tid; i < (int)(sizeof(ProblemState) / 4); i += kBlock) dst[i] = src[i];
    if (tid == 0) s_nl = P.grid->n_levels;
    if (tid < kMaxLevels) s_h[tid] = P.grid->lv[tid].h;
  }
  // step partials: each thread sums a strided subset of blocks for all four
  // coefficients, then one fixed-order tree
  __shared__ double s_b[4][kBlock];
  {
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = tid; b < nsb; b += kBlock)
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] += ld_dev(&P.part_s[(size_t)b * 4 + c]);
#pragma unroll
    for (int c = 0; c < 4; ++c) s_b[c][tid] = v[c];
  }
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    for (int t = tid; t < 4 * w; t += kBlock) {
      const int c = t / w, i = t - c * w;
      s_b[c][i] += s_b[c][i + w];
    }
    __syncthreads();
  }
  if (tid == 0) {
    for (int c = 0; c < 6; ++c) s_st.flow[c] = tot[c];
    for (int c = 0; c < 4; ++c) s_st.bcde[c] = s_b[c][0];
    if (kc.adaptive) controller_adaptive(&s_st, P.xx_st, P.yy_st, kc, P.trace, P.trace_cap, s_h, s_nl);
    else controller(&s_st, kc, P.trace, P.trace_cap, P.n_src, s_h, s_nl);
  }
  __syncthreads();
  {
    // the pass counters live at the device coherence point: never written
    // back from the staged copy; this pass's counter returns to zero
    constexpr int c0 = (int)(offsetof(ProblemState, blocks_done_assoc) / 4);
    constexpr int c1 = (int)(offsetof(ProblemState, blocks_done_step) / 4) + 1;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&s_st);
    uint32_t* dst = reinterpret_cast<uint32_t*>(st);
    for (int i = tid; i < (int)(sizeof(ProblemState) / 4); i += kBlock)
      if (i < c0 || i >= c1) dst[i] = src[i];
    if (tid == 0) st_dev(&st->blocks_done_step, 0u);
  }
}

// One thread per source row; grid (row blocks, problems).  The last block of
// a problem runs its controller step.
__device__ __forceinline__ void step_pass(const AssocProblem& P, const KConsts& kc) {
  ProblemState* st = P.st;
  if (st->done) return;
  const int tid = threadIdx.x;
  const int r = blockIdx.x * kBlock + tid;
  const int nsb = (P.n_src + kBlock - 1) / kBlock;
  if ((int)blockIdx.x >= nsb) return;  // uniform: blocks beyond this problem's rows
  double tot[6];
  scaled_flow(st, kc, tot);
  const float ell = st->ell;
  const GridLevel G = P.grid->lv[st->level];  // a register copy, as in the association
  Maps mp;
  load_maps(st, mp);
  const StepDir dir = step_direction(kc, tot);
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (r < P.n_src) {
    step_row(kc, G, mp, dir, ld_global(P.src_pos + r), ell, P.pairs + (size_t)r * P.cap_alloc,
             ld_global(P.counts + r), 0u, 1u, acc);
  }
  // block partial in fixed order: wave shuffles then LDS over the 4 waves
  __shared__ double s_w[4][kBlock / 64];
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    double v = acc[c];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) s_w[c][wave] = v;
  }
  __syncthreads();
  __shared__ int s_last;
  if (tid < 64) {
    if (tid < 4) {
      double v = 0.0;
      for (int w = 0; w < kBlock / 64; ++w) v += s_w[tid][w];
      st_dev(&P.part_s[(size_t)blockIdx.x * 4 + tid], v);
    }
    wait_stores();
    if (tid == 0) s_last = (count_in(&st->blocks_done_step) == (uint32_t)(nsb - 1)) ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;  // uniform
  controller_tail(P, kc, tot, nsb);
}

template <bool ONE>
__global__ __launch_bounds__(kBlock) void step_kernel(const AssocProblem* __restrict__ probs, KConsts kc,
                                                      AssocProblem one) {
  if constexpr (ONE) step_pass(one, kc);
  else {
    const AssocProblem P = probs[blockIdx.y];  // a register copy
    step_pass(P, kc);
  }
}

// Initial state of a problem: pose from a row-major float 4x4, maps, level.
__global__ void init_state_kernel(const AssocProblem* __restrict__ probs, int n_probs, const float* __restrict__ T16,
                                  int stride16, KConsts kc, float ell0, int K0) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_probs) return;
  const AssocProblem& P = probs[p];
  ProblemState* st = P.st;
  const float* T = T16 + (size_t)p * stride16;
  for (int r = 0; r < 3; ++r) {
    for (int c = 0; c < 3; ++c) st->R[r * 3 + c] = (double)T[r * 4 + c];
    st->T[r] = (double)T[r * 4 + 3];
  }
  for (int i = 0; i < 9; ++i) st->As[i] = (i % 4 == 0) ? 1.0f : 0.0f;
  for (int i = 0; i < 3; ++i) st->bs[i] = 0.0f;
  st->has_src_xf = 0;
  for (int c = 0; c < 6; ++c) st->flow[c] = 0.0;
  for (int c = 0; c < 4; ++c) st->bcde[c] = 0.0;
  st->ip = 0.0;
  st->step = 0.0;
  st->dist = 0.0;
  st->nnz = 0;
  st->ell = ell0;
  st->K = K0;
  st->iter = 0;
  st->done = 0;
  st->ret = 0;
  st->iters_out = 0;
  st->max_row = 0;
  st->n_overflow = 0;
  st->blocks_done_assoc = st->blocks_done_ovf = st->blocks_done_step = 0;
  st->qs_head = st->qs_size = st->qe_head = st->qe_size = 0;
  st->ss = st->se = 0.0f;
  st->ell_max = kc.ell_max0;
  st->dl = 0.0;
  set_maps(st);
  set_level(st, kc, ell0, P.grid);
}

// Switches every problem to a single scoring pass at lengthscale ell with the
// full row cap, keeping its pose (multi-start scoring by cos angle).
__global__ void rescore_state_kernel(const AssocProblem* __restrict__ probs, int n_probs, KConsts kc, float ell,
                                     int K) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_probs) return;
  const AssocProblem& P = probs[p];
  ProblemState* st = P.st;
  st->ell = ell;
  st->K = K;
  st->done = 0;
  st->n_overflow = 0;
  set_maps(st);
  set_level(st, kc, ell, P.grid);
}

// ---------------------------------------------------------------------------
// Association export: CSR in input row order, target ids ascending per row.
// ---------------------------------------------------------------------------

__global__ void export_counts(const AssocProblem* __restrict__ P, int64_t* __restrict__ counts_orig) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= P->n_src) return;
  uint32_t orig = __float_as_uint(P->src_pos[r].w);
  counts_orig[orig] = (int64_t)P->counts[r];
}

// One 64-lane wave per row: gathers (target id, a), bitonic sort by id in LDS.
// One row of the association export, sorted in LDS (bitonic, row <= 1024
// pairs) by target id, or -- for rows with more than sort_threshold pairs when
// sort_threshold > 0 -- by value descending with ties by id, the order the
// reference's multiframe_is_sorting_inner_product gives a row
// (CvoGPU.cu:1080-1095).  Keys: (id, value bits) or (~value bits, id); the
// values are positive, so their bits order like the values.
__global__ __launch_bounds__(64) void export_rows(const AssocProblem* __restrict__ P, const int64_t* __restrict__ row_ptr,
                                                  int32_t* __restrict__ col, float* __restrict__ val,
                                                  int sort_threshold) {
  __shared__ uint64_t s_key[1024];
  const int r = blockIdx.x;
  if (r >= P->n_src) return;
  const GridLevel& G = P->grid->lv[P->st->level_assoc];
  const uint32_t cnt = P->counts[r];
  const uint32_t orig = __float_as_uint(P->src_pos[r].w);
  const bool by_value = sort_threshold > 0 && cnt > (uint32_t)sort_threshold;
  uint32_t n2 = 1;
  while (n2 < cnt) n2 <<= 1;
  // bundle adjustment rows: (target coordinates, a) at the pass's row stride
  // K, the sorted target positions beside them
  const bool ba_rows = P->pairs4 != nullptr;
  const size_t row0 = ba_rows ? (size_t)r * (size_t)P->st->K : (size_t)r * P->cap_alloc;
  for (uint32_t s = threadIdx.x; s < n2; s += 64) {
    uint64_t key = ~0ull;
    if (s < cnt) {
      const uint2 e = ba_rows ? make_uint2(P->pair_ids[row0 + s], __float_as_uint(P->pairs4[row0 + s].w))
                              : P->pairs[row0 + s];
      const uint32_t id = __float_as_uint(G.pos[e.x].w);
      key = by_value ? (((uint64_t)(~e.y)) << 32) | id : (((uint64_t)id) << 32) | e.y;
    }
    s_key[s] = key;
  }
  __syncthreads();
  block_bitonic_sort(s_key, n2);
  const int64_t base = row_ptr[orig];
  for (uint32_t s = threadIdx.x; s < cnt; s += 64) {
    const uint64_t key = s_key[s];
    const uint32_t hi = (uint32_t)(key >> 32), lo = (uint32_t)key;
    col[base + s] = (int32_t)(by_value ? lo : hi);
    val[base + s] = __uint_as_float(by_value ? ~hi : lo);
  }
}

// All-done flag of a set of problems (one block), for the host's chunk loop.
__global__ void all_done_kernel(const AssocProblem* __restrict__ probs, int n_probs, int32_t* __restrict__ out) {
  __shared__ int s_any;
  if (threadIdx.x == 0) s_any = 0;
  __syncthreads();
  for (int q = threadIdx.x; q < n_probs; q += blockDim.x)
    if (!probs[q].st->done) s_any = 1;
  __syncthreads();
  if (threadIdx.x == 0) *out = s_any ? 0 : 1;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

void launch_all_done(const AssocProblem* probs, int n_probs, int32_t* out, hipStream_t s) {
  hipLaunchKernelGGL(all_done_kernel, dim3(1), dim3(256), 0, s, probs, n_probs, out);
}

// A launch, bracketed by the events e0 / e1 at the kernel's own start and end
// when e0 is given (profiling: the events time the kernel alone, as a kernel
// tracer does, not the dispatch around it).
#define CVO_LAUNCH(KERNEL, GRID, BLOCK, STREAM, E0, E1, ...)                                  \
  do {                                                                                      \
    if (E0) hipExtLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, STREAM, E0, E1, 0, __VA_ARGS__); \
    else hipLaunchKernelGGL(KERNEL, GRID, BLOCK, 0, STREAM, __VA_ARGS__);                  \
  } while (0)

template <int FC, int KC>
static void launch_assoc_t(const AssocProblem* probs, int n_probs, int total_blocks, const KConsts& kc,
                           const AssocProblem& one, bool use_one, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  const dim3 g(total_blocks), b(kBlock);
  if (kc.knn > 0) {
    if (use_one) CVO_LAUNCH((knn_assoc_kernel<FC, KC, true>), g, b, s, e0, e1, probs, n_probs, kc, one);
    else CVO_LAUNCH((knn_assoc_kernel<FC, KC, false>), g, b, s, e0, e1, probs, n_probs, kc, one);
  } else {
    if (use_one) CVO_LAUNCH((assoc_kernel<FC, KC, true>), g, b, s, e0, e1, probs, n_probs, kc, one);
    else CVO_LAUNCH((assoc_kernel<FC, KC, false>), g, b, s, e0, e1, probs, n_probs, kc, one);
  }
}

template <int FC, int KC>
static void launch_ovf_t(const AssocProblem* probs, int n_probs, const KConsts& kc, const AssocProblem& one,
                         bool use_one, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  const dim3 g(kOvfBlocks, n_probs), b(kBlock);
  if (use_one) CVO_LAUNCH((overflow_kernel<FC, KC, true>), g, b, s, e0, e1, probs, kc, one);
  else CVO_LAUNCH((overflow_kernel<FC, KC, false>), g, b, s, e0, e1, probs, kc, one);
}

static int fsel(const KConsts& kc) {
  if (!kc.use_col) return 0;
  return kc.F == 5 ? 5 : -1;
}
static int ksel(const KConsts& kc) {
  if (!kc.use_sem) return 0;
  return kc.Ks == 19 ? 19 : -1;
}

#define CVO_DISPATCH_FK(FN, ...)                              \
  do {                                                        \
    int f_ = fsel(kc), k_ = ksel(kc);                         \
    if (f_ == 0 && k_ == 0) FN<0, 0>(__VA_ARGS__);            \
    else if (f_ == 0 && k_ == 19) FN<0, 19>(__VA_ARGS__);     \
    else if (f_ == 0) FN<0, -1>(__VA_ARGS__);                 \
    else if (f_ == 5 && k_ == 0) FN<5, 0>(__VA_ARGS__);       \
    else if (f_ == 5 && k_ == 19) FN<5, 19>(__VA_ARGS__);     \
    else if (f_ == 5) FN<5, -1>(__VA_ARGS__);                 \
    else if (k_ == 0) FN<-1, 0>(__VA_ARGS__);                 \
    else if (k_ == 19) FN<-1, 19>(__VA_ARGS__);               \
    else FN<-1, -1>(__VA_ARGS__);                             \
  } while (0)

void launch_assoc(const AssocProblem* probs, int n_probs, int total_blocks, const KConsts& kc, hipStream_t s,
                  const AssocProblem* host_one, hipEvent_t e0, hipEvent_t e1) {
  AssocProblem one{};
  const bool use_one = n_probs == 1 && host_one;
  if (use_one) one = *host_one;
  CVO_DISPATCH_FK(launch_assoc_t, probs, n_probs, total_blocks, kc, one, use_one, s, e0, e1);
}

void launch_overflow(const AssocProblem* probs, int n_probs, const KConsts& kc, hipStream_t s,
                     const AssocProblem* host_one, hipEvent_t e0, hipEvent_t e1) {
  AssocProblem one{};
  const bool use_one = n_probs == 1 && host_one;
  if (use_one) one = *host_one;
  CVO_DISPATCH_FK(launch_ovf_t, probs, n_probs, kc, one, use_one, s, e0, e1);
}

void launch_step(const AssocProblem* probs, int n_probs, int max_src_rows, const KConsts& kc, hipStream_t s,
                 const AssocProblem* host_one, hipEvent_t e0, hipEvent_t e1) {
  const dim3 g((max_src_rows + kBlock - 1) / kBlock, n_probs), b(kBlock);
  AssocProblem one{};
  if (n_probs == 1 && host_one) {
    one = *host_one;
    CVO_LAUNCH(step_kernel<true>, g, b, s, e0, e1, probs, kc, one);
  } else {
    CVO_LAUNCH(step_kernel<false>, g, b, s, e0, e1, probs, kc, one);
  }
}

void launch_adaptive_sync(const AssocProblem* probs, const KConsts& kc, hipStream_t s) {
  hipLaunchKernelGGL(adaptive_sync_kernel, dim3(1), dim3(64), 0, s, probs, kc);
}

void launch_rescore(const AssocProblem* probs, int n_probs, const KConsts& kc, float ell, int K, hipStream_t s) {
  hipLaunchKernelGGL(rescore_state_kernel, dim3((n_probs + 63) / 64), dim3(64), 0, s, probs, n_probs, kc, ell, K);
}


void launch_init_state(const AssocProblem* probs, int n_probs, const float* T16, int stride16, const KConsts& kc,
                       float ell0, int K0, hipStream_t s) {
  hipLaunchKernelGGL(init_state_kernel, dim3((n_probs + 63) / 64), dim3(64), 0, s, probs, n_probs, T16, stride16, kc,
                     ell0, K0);
}

void launch_grid_count(const float* xyz, int n, const GridLevel& L, uint32_t* key, uint32_t* count, hipStream_t s) {
  hipLaunchKernelGGL(grid_cell_count, dim3((n + 255) / 256), dim3(256), 0, s, xyz, n, L.ox, L.oy, L.oz, L.inv_h, L.nx,
                     L.ny, L.nz, key, count);
}

// The controller's device math on given inputs, for checks against
// published values: the cubic (roots of coef[4i..4i+3], highest power first;
// re / im 3 each), the FP64 SE(3) exponential of dt[i] * xi[6i..] (row-major
// 3x4) with the log norm of its result, and the reference's float exponential
// of the same twist.
__global__ void math_check_kernel(int n_cubic, const double* __restrict__ coef, double* __restrict__ re,
                                  double* __restrict__ im, int n_exp, const double* __restrict__ xi,
                                  const double* __restrict__ dt, double* __restrict__ T64,
                                  double* __restrict__ log_norm, float* __restrict__ T32) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_cubic) {
    double r[3], m[3];
    cubic_solve(coef[4 * i], coef[4 * i + 1], coef[4 * i + 2], coef[4 * i + 3], r, m);
    for (int k = 0; k < 3; ++k) {
      re[3 * i + k] = r[k];
      im[3 * i + k] = m[k];
    }
  }
  if (i < n_exp) {
    double R[9], t[3];
    se3_exp(xi + 6 * i, dt[i], R, t);
    for (int r = 0; r < 3; ++r) {
      for (int c = 0; c < 3; ++c) T64[12 * i + 4 * r + c] = R[3 * r + c];
      T64[12 * i + 4 * r + 3] = t[r];
    }
    log_norm[i] = se3_log_norm(R, t);
    float xf[6];
    for (int k = 0; k < 6; ++k) xf[k] = (float)xi[6 * i + k];
    exp_sek3_f32(xf, (float)dt[i], T32 + 12 * i);
  }
}

void launch_math_check(int n_cubic, const double* coef, double* re, double* im, int n_exp, const double* xi,
                       const double* dt, double* T64, double* log_norm, float* T32, hipStream_t s) {
  const int n = n_cubic > n_exp ? n_cubic : n_exp;
  hipLaunchKernelGGL(math_check_kernel, dim3((n + 63) / 64), dim3(64), 0, s, n_cubic, coef, re, im, n_exp, xi, dt,
                     T64, log_norm, T32);
}

void launch_zero(void* p, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 4;
  if (n == 0) return;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(zero_u32, dim3((unsigned)blocks), dim3(256), 0, s, static_cast<uint32_t*>(p), n);
}

void launch_iota(uint32_t* v, int n, hipStream_t s) {
  hipLaunchKernelGGL(iota_u32, dim3((n + 255) / 256), dim3(256), 0, s, v, n);
}

void launch_gather(const uint32_t* order, int n, const float* xyz, const float* feat, int F, const float* sem, int K,
                   const float* geo, float4* pos, float* feat_s, float* sem_s, float* geo_s, uint32_t* inv_perm,
                   hipStream_t s) {
  hipLaunchKernelGGL(gather_sorted, dim3((n + 255) / 256), dim3(256), 0, s, order, n, xyz, feat, F, sem, K, geo, pos,
                     feat_s, sem_s, geo_s, inv_perm);
}

static MortonBox morton_box(const float* bmin, const float* bmax) {
  MortonBox B;
  for (int d = 0; d < 3; ++d) {
    const float ext = bmax[d] - bmin[d];
    B.o[d] = bmin[d];
    B.s[d] = ext > 0 ? 1023.0f / ext : 0.0f;
  }
  return B;
}

void launch_morton(const float* xyz, int n, const float* bmin, const float* bmax, uint32_t* key, hipStream_t s) {
  hipLaunchKernelGGL(morton_keys, dim3((n + 255) / 256), dim3(256), 0, s, xyz, n, morton_box(bmin, bmax), key);
}

static int small_padded(int n) {
  int p = 2;
  while (p < n) p <<= 1;
  return p;
}

void launch_small_source(const float* xyz, int n, const float* bmin, const float* bmax, const float* feat, int F,
                         const float* sem, int K, const float* geo, float4* pos, float* feat_s, float* sem_s,
                         float* geo_s, hipStream_t s) {
  const int padded = small_padded(n);
  hipLaunchKernelGGL(small_source_kernel, dim3(1), dim3(1024), sizeof(uint64_t) * padded, s, xyz, n, padded,
                     morton_box(bmin, bmax), pos);
  if (feat_s || sem_s || geo_s)
    hipLaunchKernelGGL(small_attributes_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, pos, feat, F, sem, K, geo,
                       feat_s, sem_s, geo_s);
}

// G's levels hold their arrays' addresses.
void launch_small_levels(const float* xyz, int n, const GridDev& G, uint32_t max_cells, const float* feat, int F,
                         const float* sem, int K, const float* geo, hipStream_t s) {
  const int padded = small_padded(n), pb = (n + 255) / 256;
  hipLaunchKernelGGL(small_levels_kernel, dim3(G.n_levels), dim3(1024), sizeof(uint64_t) * padded, s, xyz, n, padded, G);
  const unsigned cb = (unsigned)(((size_t)max_cells + 1 + kCellsPerBlock - 1) / kCellsPerBlock);
  hipLaunchKernelGGL(small_cells_kernel, dim3(pb + cb, G.n_levels), dim3(256), 0, s, n, pb, G, feat, F, sem, K, geo);
}

void launch_export(const AssocProblem* P_dev, int n_src, int64_t* counts_orig, const int64_t* row_ptr, int32_t* col,
                   float* val, int phase, int sort_threshold, hipStream_t s) {
  if (phase == 0)
    hipLaunchKernelGGL(export_counts, dim3((n_src + 255) / 256), dim3(256), 0, s, P_dev, counts_orig);
  else
    hipLaunchKernelGGL(export_rows, dim3(n_src), dim3(64), 0, s, P_dev, row_ptr, col, val, sort_threshold);
}

}  // namespace cvo
