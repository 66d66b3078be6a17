// Multifrontal LU of the components too large for the task lists of
// xg_lu.hip (the 20k-node random logic, the 550k-unknown power grid): the
// refactor-and-solve that replaces N_LAS_AmesosSolver::solve (KLU,
// N_LAS_AmesosSolver.C:231-470) for them.
//
// The plan (xg_lu_setup.cpp) gives every component a tree of dense fronts:
// front s owns k consecutive pivot positions (its fully summed columns)
// and has m >= k rows; its m x m block is row-major in one value buffer.
// Per Newton iteration:
//  1. every front is cleared and the Jacobian's entries are scattered into
//     the fronts that own them; the right-hand side is one more column of
//     each front (its fully summed rows' entries, zero below);
//  2. level by level from the leaves (a level's fronts are independent),
//     a front adds its children's contribution blocks (in child order), then
//     factors its k fully summed columns: blocked right-looking LU, pivots
//     chosen by magnitude among the fully summed rows only, the trailing
//     update leaving the Schur complement (the contribution block) in the
//     bottom-right corner.  The right-hand-side column takes the same swaps
//     and updates, so the forward solve is done when the factorisation is,
//     and L is not kept;
//  3. the backward solve walks the levels back down;
// Updates go by groups of four pivots (aligned in the front): a group's
// products for an element are summed from zero, by fused multiply-adds in
// ascending order, and the sum is added; within the group's own rows and
// columns each is subtracted at once.  Every form below does exactly that, so
// all forms give an element the same bits.  One chain over all pivots rounds
// at the element's full size every time: on power grids, whose rows nearly
// cancel, its solutions were 1.2 to 1.4 times as far from the exact one.
//  4. one workgroup per component checks the normwise backward error
//     against the unfactored rows, applies x += dx and forms the weighted
//     RMS norm, as the task-list kernel does.
// Every sum is in a fixed order, so the results do not depend on the
// launch.  A pivot column with no nonzero candidate, or a backward error
// above the bound, hands the component to the dense partial-pivoting
// kernel (as the task lists do); beyond that kernel's size it stays
// singular (stats[2] = 1) with its iterate unchanged.
#include <algorithm>
#include <cfloat>

#include "xg_internal.h"
#include "xg_lu_dev.h"

namespace xg {

namespace {

constexpr int kFB = 256;           // threads per front workgroup
constexpr int kFinishBlock = 1024;  // threads of the per-component check
constexpr int kSolveBlock = 512;    // threads of a solve workgroup for fronts above 512 rows

// (value, smallest index) maximum over the block: per wavefront, then
// across the B / 64 wavefronts.
template <int B>
__device__ __forceinline__ void blk_argmax(double v, int idx, double *sv, int *si,
                                           double &best, int &bi) {
  for (int off = 32; off >= 1; off >>= 1) {
    const double ov = __shfl_xor(v, off);
    const int oi = __shfl_xor(idx, off);
    if (ov > v || (ov == v && oi < idx)) {
      v = ov;
      idx = oi;
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    sv[w] = v;
    si[w] = idx;
  }
  __syncthreads();
  best = sv[0];
  bi = si[0];
  for (int q = 1; q < B / 64; ++q)
    if (sv[q] > best || (sv[q] == best && si[q] < bi)) {
      best = sv[q];
      bi = si[q];
    }
  __syncthreads();
}

template <int B>
__device__ __forceinline__ double blk_reduce(double v, double *sv, bool is_max) {
  const int t = threadIdx.x;
  sv[t] = v;
  __syncthreads();
  for (int s = B / 2; s > 0; s >>= 1) {
    if (t < s) sv[t] = is_max ? fmax(sv[t], sv[t + s]) : sv[t] + sv[t + s];
    __syncthreads();
  }
  const double r = sv[0];
  __syncthreads();
  return r;
}

// Partial LU of the m x m row-major front A and its right-hand side w (the
// virtual column m): its first k columns, pivots among rows [j, k) for
// column j.  Panels of NB columns factor in the LDS buffer P (rows
// kb..m-1, stride NB + 1); the panel's row swaps are then applied to the
// columns right of it, U12 is solved column by column in registers and the
// trailing block takes the panel's rank-NB update.  Every sum of products
// runs over groups of four pivots, as described at the top.  False when a
// pivot column has no nonzero candidate.
template <int NB, int BS = kFB>
__device__ bool front_factor(double *A, double *w, int m, int k, double *P, double *sv,
                             int *si, int *spiv) {
  const int t = threadIdx.x;
  constexpr int PS = NB + 1;
  for (int kb = 0; kb < k; kb += NB) {
    const int nb = min(NB, k - kb);
    const int rows = m - kb;      // panel rows
    const int cand = k - kb;      // rows eligible as pivots
    for (int e = t; e < rows * NB; e += BS) {
      const int r = e / NB, c = e % NB;
      P[r * PS + c] = c < nb ? A[(int64_t)(kb + r) * m + kb + c] : 0.0;
    }
    __syncthreads();
    for (int c = 0; c < nb; ++c) {
      double v = -1.0;
      int idx = 0x7fffffff;
      for (int r = c + t; r < cand; r += BS) {
        const double a = fabs(P[r * PS + c]);
        if (a > v) {
          v = a;
          idx = r;
        }
      }
      double best;
      int br;
      blk_argmax<BS>(v, idx, sv, si, best, br);
      if (!(best > 0.0) || !(best <= DBL_MAX)) return false;  // same on every thread
      if (t == 0) spiv[c] = kb + br;
      if (br != c)
        for (int cc = t; cc < NB; cc += BS) {
          const double tmp = P[c * PS + cc];
          P[c * PS + cc] = P[br * PS + cc];
          P[br * PS + cc] = tmp;
        }
      __syncthreads();
      const Pivot pv = make_pivot(P[c * PS + c]);
      const int g0 = c & ~3, g1 = min(g0 + 4, nb);  // the column's group
      for (int r = c + 1 + t; r < rows; r += BS) {
        const double l = divide(P[r * PS + c], pv);
        P[r * PS + c] = l;
        for (int cc = c + 1; cc < g1; ++cc)
          P[r * PS + cc] = fma(-l, P[c * PS + cc], P[r * PS + cc]);
      }
      __syncthreads();
      if (c + 1 < g1 || g1 == nb) continue;
      // the group's rows of U, then its products for the rows below
      for (int cc = g1 + t; cc < nb; cc += BS)
        for (int i = g0 + 1; i < g1; ++i)
          for (int j = g0; j < i; ++j)
            P[i * PS + cc] = fma(-P[i * PS + j], P[j * PS + cc], P[i * PS + cc]);
      __syncthreads();
      for (int r = g1 + t; r < rows; r += BS)
        for (int cc = g1; cc < nb; ++cc) {
          double p = 0.0;
          for (int j = g0; j < g1; ++j) p = fma(-P[r * PS + j], P[j * PS + cc], p);
          P[r * PS + cc] = P[r * PS + cc] + p;
        }
      __syncthreads();
    }
    for (int e = t; e < nb * NB; e += BS) {  // U11 (and L11, unused later)
      const int r = e / NB, c = e % NB;
      if (c < nb) A[(int64_t)(kb + r) * m + kb + c] = P[r * PS + c];
    }
    const int j0 = kb + nb, ncols = m + 1 - j0;
    // column j of the front, j = m the right-hand side
    auto col = [&](int j, int64_t &ld) {
      ld = j < m ? m : 1;
      return j < m ? A + j : w;
    };
    // the panel's row swaps on the columns right of it, in pivot order
    for (int j = j0 + t; j <= m; j += BS) {
      int64_t ld;
      double *a = col(j, ld);
      for (int c = 0; c < nb; ++c) {
        const int pr = spiv[c];
        if (pr != kb + c) {
          const double tmp = a[(kb + c) * ld];
          a[(kb + c) * ld] = a[pr * ld];
          a[pr * ld] = tmp;
        }
      }
    }
    __syncthreads();
    // U12 of column j (rows kb..kb+nb-1) by the unit lower panel block
    auto solve_u = [&](const double *a, int64_t ld, double *u) {
#pragma unroll
      for (int c = 0; c < NB; ++c) u[c] = c < nb ? a[(kb + c) * ld] : 0.0;
#pragma unroll
      for (int g = 0; g < NB; g += 4) {
#pragma unroll
        for (int c = g; c < g + 4; ++c)
#pragma unroll
          for (int i = c + 1; i < g + 4; ++i)
            if (i < nb) u[i] = fma(-P[i * PS + c], u[c], u[i]);
#pragma unroll
        for (int i = g + 4; i < NB; ++i)
          if (i < nb) {
            double p = 0.0;
#pragma unroll
            for (int c = g; c < g + 4; ++c) p = fma(-P[i * PS + c], u[c], p);
            u[i] = u[i] + p;
          }
      }
    };
    // rows j0+g, j0+g+G, ... of a column take the panel's updates
    auto sweep = [&](double *a, int64_t ld, int g, int G, const double *u) {
      for (int i = j0 + g; i < m; i += 4 * G) {
        double x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int ii = i + q * G;
          x[q] = ii < m ? a[ii * ld] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int ii = i + q * G;
          if (ii < m) {
            const double *l = P + (ii - kb) * PS;
            double v = x[q];
#pragma unroll
            for (int g = 0; g < NB; g += 4)
              if (g < nb) {
                double p = 0.0;
#pragma unroll
                for (int c = g; c < g + 4; ++c)
                  if (c < nb) p = fma(-l[c], u[c], p);
                v = v + p;
              }
            a[ii * ld] = v;
          }
        }
      }
    };
    if (ncols >= BS) {
      for (int j = j0 + t; j <= m; j += BS) {
        int64_t ld;
        double *a = col(j, ld);
        double u[NB];
        solve_u(a, ld, u);
#pragma unroll
        for (int c = 0; c < NB; ++c)
          if (c < nb) a[(kb + c) * ld] = u[c];
        sweep(a, ld, 0, 1, u);
      }
    } else {
      const int G = min(BS / ncols, 16);
      const bool mine = t < ncols * G;
      const int g = t / ncols;
      int64_t ld;
      double *a = col(j0 + t % ncols, ld);
      double u[NB];
      if (mine) solve_u(a, ld, u);
      __syncthreads();
      if (mine) {
        if (g == 0)
#pragma unroll
          for (int c = 0; c < NB; ++c)
            if (c < nb) a[(kb + c) * ld] = u[c];
        sweep(a, ld, g, G, u);
      }
    }
    __syncthreads();
  }
  return true;
}

__device__ __forceinline__ bool front_skip(const FrontArgs &f, int c) {
  return (f.gate && *f.gate) || (f.active && !f.active[c]) || f.bad[c];
}

// The same for a workgroup of a launch that sets the flag: another front of
// component c, in the same launch, can fail while this workgroup's
// wavefronts start, and wavefronts that read different values would leave some
// of them running with LDS that the others never wrote.  So one thread reads
// it for all of them.
__device__ __forceinline__ bool front_skip_block(const FrontArgs &f, int c, int *flag) {
  if (threadIdx.x == 0) *flag = front_skip(f, c);
  __syncthreads();
  return *flag != 0;
}

// Clears the fronts and the failure flags and sets the right-hand-side
// columns, then (second kernel) scatters the Jacobian's entries.
__global__ void __launch_bounds__(kFB) front_clear_kernel(FrontArgs f, const double *bp) {
  if (f.gate && *f.gate) return;
  const int64_t stride = (int64_t)gridDim.x * kFB;
  for (int64_t i = (int64_t)blockIdx.x * kFB + threadIdx.x; i < f.n_vals; i += stride)
    f.vals[i] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kFB + threadIdx.x; i < f.n_rows; i += stride) {
    const int32_t r = f.rsrc[i];
    f.wrhs[i] = r >= 0 ? bp[r] : 0.0;
  }
  for (int64_t i = (int64_t)blockIdx.x * kFB + threadIdx.x; i < f.n_comp; i += stride)
    f.bad[i] = 0;
}

__global__ void __launch_bounds__(kFB) front_scatter_kernel(FrontArgs f, const double *J) {
  if (f.gate && *f.gate) return;
  const int64_t stride = (int64_t)gridDim.x * kFB;
  for (int64_t e = (int64_t)blockIdx.x * kFB + threadIdx.x; e < f.n_ent; e += stride)
    f.vals[f.ent_fpos[e]] = J[f.ent_k[e]];
}

template <int NB, int ROWS, int BS>
__global__ void __launch_bounds__(BS) front_factor_kernel(FrontArgs f, int lv0) {
  __shared__ double P[ROWS * (NB + 1)];
  __shared__ double sv[BS / 64];
  __shared__ int si[BS / 64];
  __shared__ int spiv[NB], skip;
  const int s = f.lv[lv0 + blockIdx.x];
  const int c = f.comp[s];
  if (front_skip_block(f, c, &skip)) return;
  const int t = threadIdx.x;
  const int m = f.m[s], k = f.k[s];
  if (m > f.big_m) return;  // factored by many workgroups (launch_big_front)
  double *A = f.vals + f.fo[s], *w = f.wrhs + f.ro[s];
  // the children's contribution blocks, in child order
  for (int q = f.ch_ptr[s]; q < f.ch_ptr[s + 1]; ++q) {
    const int ch = f.ch[q];
    const int mc = f.m[ch], kc = f.k[ch], wc = mc - kc;
    const double *C = f.vals + f.fo[ch] + (int64_t)kc * mc + kc;
    const double *r = f.wrhs + f.ro[ch] + kc;
    const int32_t *map = f.cbmap + f.ro[ch] + kc;
    for (int64_t e = t; e < (int64_t)wc * wc; e += BS) {
      const int i = (int)(e / wc), j = (int)(e % wc);
      A[(int64_t)map[i] * m + map[j]] += C[(int64_t)i * mc + j];
    }
    for (int i = t; i < wc; i += BS) w[map[i]] += r[i];
    __syncthreads();
  }
  if (!front_factor<NB, BS>(A, w, m, k, P, sv, si, spiv))
    if (t == 0) f.bad[c] = 1;
}

// Fronts of up to kTinyM rows, one thread each (a level of the tree's
// bottom holds up to ~10^5 of them): the children's contribution blocks in
// child order, then the LU by groups of four columns with whole-row swaps,
// pivots among the fully summed rows (largest magnitude, smallest index on
// ties).  Every element takes the same operations in the same order as in the
// other forms, so all give the same bits.

__global__ void __launch_bounds__(64) front_tiny_kernel(FrontArgs f, int lv0, int nfr) {
  const int q = blockIdx.x * 64 + threadIdx.x;
  if (q >= nfr) return;
  const int s = f.lv[lv0 + q];
  const int c = f.comp[s];
  if (front_skip(f, c)) return;
  const int m = f.m[s], k = f.k[s];
  if (m > f.big_m) return;
  double *A = f.vals + f.fo[s], *w = f.wrhs + f.ro[s];
  for (int qq = f.ch_ptr[s]; qq < f.ch_ptr[s + 1]; ++qq) {
    const int ch = f.ch[qq];
    const int mc = f.m[ch], kc = f.k[ch], wc = mc - kc;
    const double *C = f.vals + f.fo[ch] + (int64_t)kc * mc + kc;
    const double *r = f.wrhs + f.ro[ch] + kc;
    const int32_t *map = f.cbmap + f.ro[ch] + kc;
    for (int i = 0; i < wc; ++i) {
      for (int j = 0; j < wc; ++j) A[map[i] * m + map[j]] += C[i * mc + j];
      w[map[i]] += r[i];
    }
  }
  for (int g0 = 0; g0 < k; g0 += 4) {
    const int g1 = min(g0 + 4, k);
    for (int col = g0; col < g1; ++col) {
      double best = -1.0;
      int br = col;
      for (int r = col; r < k; ++r) {
        const double a = fabs(A[r * m + col]);
        if (a > best) {
          best = a;
          br = r;
        }
      }
      if (!(best > 0.0) || !(best <= DBL_MAX)) {
        f.bad[c] = 1;
        return;
      }
      if (br != col) {  // (with the group's multipliers)
        for (int j = g0; j < m; ++j) {
          const double tmp = A[col * m + j];
          A[col * m + j] = A[br * m + j];
          A[br * m + j] = tmp;
        }
        const double tmp = w[col];
        w[col] = w[br];
        w[br] = tmp;
      }
      const Pivot pv = make_pivot(A[col * m + col]);
      for (int r = col + 1; r < m; ++r) {
        const double l = divide(A[r * m + col], pv);
        A[r * m + col] = l;
        for (int j = col + 1; j < g1; ++j) A[r * m + j] = fma(-l, A[col * m + j], A[r * m + j]);
      }
    }
    for (int j = g1; j <= m; ++j) {  // the other columns, m the right-hand side
      double *a = j < m ? A + j : w;
      const int ld = j < m ? m : 1;
      double u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (g0 + i >= g1) continue;
        u[i] = a[(g0 + i) * ld];
#pragma unroll
        for (int q = 0; q < i; ++q) u[i] = fma(-A[(g0 + i) * m + g0 + q], u[q], u[i]);
        a[(g0 + i) * ld] = u[i];
      }
      for (int r = g1; r < m; ++r) {
        double p = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (g0 + q < g1) p = fma(-A[r * m + g0 + q], u[q], p);
        a[r * ld] = a[r * ld] + p;
      }
    }
  }
}

// ---- many-workgroup form of the large fronts (rows m > big_m), all of a
// level's at once (blockIdx.y or .z = the front among the level's large
// ones, f.big[lb + that]).  Per panel of up to kBigW fully summed columns:
//  panel    one workgroup per front factors the panel's fully summed rows
//           (the only pivot candidates);
//  solve    the columns right of it, the right-hand side included, take the
//           panel's row swaps and their U12 rows (a lane per column), and
//           the rows below the fully summed block their L21 (a lane per
//           row): one launch, 64-lane workgroups;
//  update   the trailing block takes the rank-kBigW update, 64 x 64 tiles on
//           the FP64 matrix cores.
// A front whose columns are all factored leaves the later launches at once.
constexpr int kTile = 64;   // trailing-update tile

// The children's contribution blocks, one workgroup per receiving row of
// a front (blockIdx.x = the row among the front's receiving rows): the
// child rows that land on it, in child order, each added across its
// columns and the right-hand side, so every element takes its children's
// terms in child order.
__global__ void __launch_bounds__(kFB) front_extend_kernel(FrontArgs f, int lb) {
  const BigFront s = f.big[lb + blockIdx.y];
  if (front_skip(f, s.comp)) return;
  const int64_t q = s.xr0 + blockIdx.x;
  if (q >= s.xr1) return;
  const int m = s.m;
  const int row = f.xr_row[q];
  double *Ar = f.vals + s.fo + (int64_t)row * m;
  double *wr = f.wrhs + s.ro + row;
  for (int64_t e = f.ext_ptr[q]; e < f.ext_ptr[q + 1]; ++e) {
    const int ch = f.ext_ch[e], i = f.ext_i[e];
    const int mc = f.m[ch], kc = f.k[ch], w = mc - kc;
    const double *C = f.vals + f.fo[ch] + (int64_t)(kc + i) * mc + kc;
    const int32_t *map = f.cbmap + f.ro[ch] + kc;
    for (int j = threadIdx.x; j < w; j += kFB) Ar[map[j]] += C[j];
    if (threadIdx.x == 0) *wr += f.wrhs[f.ro[ch] + kc + i];
    __syncthreads();
  }
}

// Maximum of a word over lanes 0 .. 63 (kSteps = 6) or 0 .. 2^kSteps - 1, from
// that range's last lane: row shifts, then the row broadcasts, each folded
// into one v_max_u32.
template <int kCtrl, int kRows>
__device__ __forceinline__ unsigned dpp_max(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRows, 0xf, false);
  return o > v ? o : v;
}
template <int kSteps>
__device__ __forceinline__ unsigned lanes_max(unsigned v) {
  if (kSteps > 0) v = dpp_max<0x111, 0xf>(v);
  if (kSteps > 1) v = dpp_max<0x112, 0xf>(v);
  if (kSteps > 2) v = dpp_max<0x114, 0xf>(v);
  if (kSteps > 3) v = dpp_max<0x118, 0xf>(v);
  if (kSteps > 4) v = dpp_max<0x142, 0xa>(v);
  if (kSteps > 5) v = dpp_max<0x143, 0xc>(v);
  return (unsigned)__builtin_amdgcn_readlane((int)v, (1 << kSteps) - 1);
}
// The lane (of the first 2^kSteps) with the largest v >= 0, the smallest p
// on ties (lanes holding no candidate: v = 0, which never wins over one).
// Magnitudes order as their bits do: the high words first, the low ones
// only where several high words tie.
template <int kSteps>
__device__ __forceinline__ int lane_of_max(double v, int p) {
  constexpr unsigned long long kLanes = kSteps > 5 ? ~0ull : (1ull << (1 << kSteps)) - 1;
  const unsigned hi = (unsigned)__double2hiint(v), lo = (unsigned)__double2loint(v);
  const unsigned mh = lanes_max<kSteps>(hi);
  unsigned long long mask = __ballot(hi == mh) & kLanes;
  if (mask & (mask - 1)) {
    const unsigned ml = lanes_max<kSteps>(hi == mh ? lo : 0u);
    mask = __ballot(hi == mh && lo == ml) & kLanes;
    if (mh | ml) {
      int lane = __ffsll(mask) - 1;
      int best = __builtin_amdgcn_readlane(p, lane);
      for (mask &= mask - 1; mask; mask &= mask - 1) {
        const int b = __ffsll(mask) - 1;
        const int o = __builtin_amdgcn_readlane(p, b);
        if (o < best) {
          best = o;
          lane = b;
        }
      }
      return lane;
    }
  }
  return __ffsll(mask) - 1;
}

// One panel: columns [kb, kb + W) of the rows [kb, k), W = 16 kCT.  The panel
// stays in registers as 16 x 16 tiles in the layout of the FP64 matrix cores
// (below), kNT tiles of rows per wavefront.  Four columns at a time go
// through LDS to one row per lane (kNT / 4 rows), where a column step is:
// the largest candidate of the wavefront by DPP, each wavefront's candidate
// row of four to LDS, one barrier, then every lane takes the best one and
// updates its rows' four columns.  The remaining columns then take the four
// pivot rows' U (solved by every lane for its column) and one rank-4 product
// per tile.  Rows are not moved: a lane tracks the position its row has
// after the swaps (ties go to the smallest position, as in the other forms).
// Finished pivot rows go to their position of A; the multipliers go to the
// column-major panel buffer by original row, with f.piv the original row of
// each position and f.mv the rows displaced from the panel's block.
// What bounds it is a column step's chain (~700 cycles: two searches of 200,
// the exchange through LDS of 300, the division).  With whole rows of 32 in
// lanes the exchange of a row (32 b128 LDS operations of ~40 cycles each)
// took 4000 cycles a column.
typedef double double4v __attribute__((ext_vector_type(4)));

// acc + the four products of a group, summed from zero.
__device__ __forceinline__ double4v add_group(double a, double b, const double4v &acc) {
  const double4v p = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, double4v{0.0, 0.0, 0.0, 0.0},
                                                          0, 0, 0);
  return {acc[0] + p[0], acc[1] + p[1], acc[2] + p[2], acc[3] + p[3]};
}

// What a panel's wavefronts exchange in a group of four columns: their
// candidates (value, reciprocal, position, row) and candidate rows' entries of
// these columns, two groups deep.
template <int NW>
struct PanelLds {
  double srow[2][4][NW][4];
  double sval[2][4][NW], srcp[2][4][NW];
  int spos[2][4][NW], sphy[2][4][NW], nmove;
};

// The column steps of one group, a row's entries of its four columns per lane
// (a; R rows each, at positions pos): ln gets minus the multipliers, L their
// columns, A the pivot rows' entries, win each pivot row's wavefront (four
// bits each).  False when a column has no pivot.
template <int NW, int R>
__device__ __forceinline__ bool panel_columns(PanelLds<NW> &sh, int par, int c0, int nw, int wrow,
                                              double (&a)[R][4], double (&ln)[R][4],
                                              int (&pos)[R], double *A, double *L, int m,
                                              int32_t *mv, unsigned &win) {
  constexpr int kSteps = NW >= 16 ? 4 : NW >= 8 ? 3 : NW >= 4 ? 2 : 1;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  win = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = c0 + j;
    if (c >= nw) continue;
    double v = 0.0, x0 = 0.0;
    int p = 0x7fffffff, qb = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double x = fabs(a[q][j]);
      if (pos[q] >= c && (x > v || (x == v && pos[q] < p))) {
        v = x;
        x0 = a[q][j];
        p = pos[q];
        qb = q;
      }
    }
    // the reciprocal every lane's candidate would need, while the
    // search below waits on its chain
    double rcp = make_pivot(x0).r;
    const int wl = lane_of_max<6>(v, p);
    if (lane == wl) {
      sh.sval[par][j][wave] = v;
      sh.srcp[par][j][wave] = rcp;
      sh.spos[par][j][wave] = p;
      sh.sphy[par][j][wave] = wrow + 64 * qb + lane;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        double x = a[0][jj];
#pragma unroll
        for (int q = 1; q < R; ++q) {
          double aq = a[q][jj];
          asm("" : "+v"(aq));  // a select of values, not an indexed load
          x = qb == q ? aq : x;
        }
        sh.srow[par][j][wave][jj] = x;
      }
    }
    int bw = 0;
    double best;
    if constexpr (NW == 1) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      best = sh.sval[par][j][0];
    } else {
      __syncthreads();
      // the best wavefront: lanes 0..NW-1 hold the candidates
      const double cv = lane < NW ? sh.sval[par][j][lane] : 0.0;
      const int cp = lane < NW ? sh.spos[par][j][lane] : 0x7fffffff;
      bw = lane_of_max<kSteps>(cv, cp);
      best = read_lane(cv, bw);
    }
    if (!(best > 0.0) || !(best <= DBL_MAX)) {  // the same in every lane
      if (threadIdx.x == 0) mv[0] = -1;  // the solve launch flags the component
      return false;
    }
    win |= (unsigned)bw << (4 * j);
    const int bp = sh.spos[par][j][bw];
    double u[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) u[jj] = sh.srow[par][j][bw][jj];
    const Pivot pv{__builtin_amdgcn_frexp_mant(u[j]), sh.srcp[par][j][bw],
                   -__builtin_amdgcn_frexp_exp(u[j])};
    // the finished pivot row's entries of these columns
    if (wave == 0 && lane >= j && lane < 4 && c0 + lane < nw)
      A[(int64_t)c * m + c0 + lane] = sh.srow[par][j][bw][lane];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      pos[q] = pos[q] == bp ? c : (pos[q] == c ? bp : pos[q]);
      if (pos[q] > c) {
        const double l = divide(a[q][j], pv);
        L[(int64_t)c * m + wrow + 64 * q + lane] = l;
        a[q][j] = l;
        ln[q][j] = -l;
#pragma unroll
        for (int jj = j + 1; jj < 4; ++jj) a[q][jj] = fma(-l, u[jj], a[q][jj]);
      }
    }
  }
  return true;
}

// The rows at each position after a panel, and those displaced from its block.
template <int NW, int R>
__device__ __forceinline__ void panel_rows(PanelLds<NW> &sh, const int (&pos)[R], int wrow,
                                           int nw, int kb, int32_t *piv, int32_t *mv) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = wrow + 64 * q + lane;
    if (pos[q] >= 0) {
      piv[pos[q]] = kb + r;
      if (pos[q] >= nw && pos[q] != r) {
        const int e = atomicAdd(&sh.nmove, 1);  // at most nw rows
        mv[1 + 2 * e] = kb + pos[q];
        mv[2 + 2 * e] = kb + r;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) mv[0] = sh.nmove;
}

template <int NW, int kNT, int kCT>
__global__ void __launch_bounds__(NW * 64) front_panel_kernel(FrontArgs f, int lb, int kb) {
  constexpr int R = kNT / 4, W = 16 * kCT, kRows = 16 * kNT;
  static_assert(kNT % 4 == 0 && NW <= 16 && (NW & (NW - 1)) == 0, "rows per lane, search");
  __shared__ __align__(16) double S[NW][kRows][4];
  __shared__ __align__(16) PanelLds<NW> sh;
  __shared__ double raw[4][W];
  const BigFront s = f.big[lb + blockIdx.x];
  // (no workgroup of this launch sets f.bad, so every wavefront reads the same)
  if (front_skip(f, s.comp)) return;
  const int m = s.m, k = s.k;
  if (kb >= k) return;
  const int nw = min(W, k - kb), nr = k - kb;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wrow = wave * kRows;
  double *A = f.vals + s.fo + (int64_t)kb * m + kb;
  double *L = f.lbuf + s.lo + kb;  // column c: L + c m
  int32_t *mv = f.mv + (int64_t)blockIdx.x * kMoveInts;
  if (threadIdx.x == 0) sh.nmove = 0;  // (used behind the columns' barriers)
  double4v acc[kNT][kCT];
#pragma unroll
  for (int t = 0; t < kNT; ++t)
#pragma unroll
    for (int c = 0; c < kCT; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = wrow + 16 * t + lk + 4 * r, j = 16 * c + li;
        acc[t][c][r] = load_if((i < nr) & (j < nw), A, (int64_t)i * m + j);
      }
  int pos[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = wrow + 64 * q + lane;
    pos[q] = r < nr ? r : -1;
  }
#pragma unroll
  for (int ct = 0; ct < kCT; ++ct) {
#pragma unroll 1
    for (int s4 = 0; s4 < 4; ++s4) {  // (one copy: the code must stay in the cache)
      const int c0 = 16 * ct + 4 * s4;
      if (c0 >= nw) break;
      const int par = s4 & 1;
      // four columns to one row per lane
      if ((li >> 2) == s4)
#pragma unroll
        for (int t = 0; t < kNT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[wave][16 * t + lk + 4 * r][li & 3] = acc[t][ct][r];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      double a[R][4], ln[R][4];
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[q][j] = S[wave][64 * q + lane][j];
          ln[q][j] = -0.0;
        }
      unsigned win;  // the wavefront of each pivot row, four bits each
      if (!panel_columns(sh, par, c0, nw, wrow, a, ln, pos, A, L, m, mv, win)) return;
      if (c0 + 4 >= nw) break;
      // the four pivot rows' other columns, from the lanes that hold them
#pragma unroll 1
      for (int j = 0; j < 4; ++j) {
        const int ph =
            __builtin_amdgcn_readfirstlane(sh.sphy[par][j][win >> (4 * j) & 15]) - wrow;
        if (ph < 0 || ph >= kRows) continue;
#pragma unroll
        for (int t = 0; t < kNT; ++t)
          if ((ph >> 4) == t) {
            const int r = (ph >> 2) & 3;
#pragma unroll
            for (int q = ct; q < kCT; ++q) {
              const double4v x = acc[t][q];
              const double y = r == 0 ? x[0] : r == 1 ? x[1] : r == 2 ? x[2] : x[3];
              if (lk == (ph & 3)) raw[j][16 * q + li] = y;
            }
            asm volatile("; tile %0" ::"n"(t));  // (kept apart: fixed registers)
          }
      }
      if constexpr (NW == 1) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      } else {
        __syncthreads();
      }
      double ub[kCT];
#pragma unroll
      for (int q = ct; q < kCT; ++q) {
        double u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          u[j] = raw[j][16 * q + li];
#pragma unroll
          for (int i = 0; i < j; ++i) u[j] = fma(-sh.srow[par][j][win >> (4 * j) & 15][i], u[i], u[j]);
        }
        const int col = 16 * q + li;
        const double x = lk == 0 ? u[0] : lk == 1 ? u[1] : lk == 2 ? u[2] : u[3];
        ub[q] = col >= c0 + 4 ? x : 0.0;
        if (wave == 0 && col >= c0 + 4 && col < nw) A[(int64_t)(c0 + lk) * m + col] = x;
      }
#pragma unroll
      for (int q = 0; q < R; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) S[wave][64 * q + lane][j] = ln[q][j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < kNT; ++t) {
        const double av = S[wave][16 * t + li][lk];
#pragma unroll
        for (int q = ct; q < kCT; ++q)
          acc[t][q] = add_group(av, ub[q], acc[t][q]);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  panel_rows(sh, pos, wrow, nw, kb, f.piv + s.ro + kb, mv);
}

// The same for more rows than the registers hold (above 2048): the panel's 16
// columns wait in the panel buffer, a column's place until its multipliers
// take it, and a group's products are added to them there, a row per lane.
// In registers, 28 row tiles a wavefront, the compiler spilled 319 of them: a
// 3440-row front took 26.5 ms, here 20.9.
template <int NW, int R>
__global__ void __launch_bounds__(NW * 64) front_tall_panel_kernel(FrontArgs f, int lb, int kb) {
  constexpr int W = 16;
  static_assert(kFrontMaxM <= NW * 64 * R, "rows of the tallest panel");
  __shared__ __align__(16) PanelLds<NW> sh;
  __shared__ double U[4][W];
  const BigFront s = f.big[lb + blockIdx.x];
  // (no workgroup of this launch sets f.bad, so every wavefront reads the same)
  if (front_skip(f, s.comp)) return;
  const int m = s.m, k = s.k;
  if (kb >= k) return;
  const int nw = min(W, k - kb), nr = k - kb;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wrow = wave * 64 * R;
  double *A = f.vals + s.fo + (int64_t)kb * m + kb;
  double *L = f.lbuf + s.lo + kb;  // column c: L + c m
  int32_t *mv = f.mv + (int64_t)blockIdx.x * kMoveInts;
  if (threadIdx.x == 0) sh.nmove = 0;  // (used behind the columns' barriers)
  int pos[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = wrow + 64 * q + lane;
    pos[q] = r < nr ? r : -1;
  }
  // rows of A to the buffer's columns, a quarter wavefront along a row
  {
    const int li = lane & 15;
#pragma unroll 4
    for (int r = wrow + (lane >> 4); r < min(wrow + 64 * R, nr); r += 4)
      if (li < nw) L[(int64_t)li * m + r] = A[(int64_t)r * m + li];
  }
  __syncthreads();
#pragma unroll 1
  for (int c0 = 0; c0 < nw; c0 += 4) {
    const int par = (c0 >> 2) & 1;
    double a[R][4], ln[R][4];
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[q][j] = load_if((pos[q] >= 0) & (c0 + j < nw), L,
                          (int64_t)(c0 + j) * m + wrow + 64 * q + lane);
        ln[q][j] = -0.0;
      }
    unsigned win;
    if (!panel_columns(sh, par, c0, nw, wrow, a, ln, pos, A, L, m, mv, win)) return;
    const int nc = nw - c0 - 4;  // the columns after the group
    if (nc <= 0) break;
    // the four pivot rows' entries of them (complete: the columns' barriers
    // lie behind the last group's sums), a column per lane
    if (threadIdx.x < nc) {
      const int col = c0 + 4 + threadIdx.x;
      double u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        u[j] = L[(int64_t)col * m + sh.sphy[par][j][win >> (4 * j) & 15]];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < j; ++i)
          u[j] = fma(-sh.srow[par][j][win >> (4 * j) & 15][i], u[i], u[j]);
        U[j][threadIdx.x] = u[j];
        A[(int64_t)(c0 + j) * m + col] = u[j];
      }
    }
    __syncthreads();
#pragma unroll 2
    for (int c = 0; c < nc; ++c) {
      double *Lc = L + (int64_t)(c0 + 4 + c) * m + wrow + lane;
      double x[R];
#pragma unroll
      for (int q = 0; q < R; ++q) x[q] = load_if(pos[q] > c0 + 3, Lc, 64 * q);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        double p = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) p = fma(ln[q][j], U[j][c], p);
        if (pos[q] > c0 + 3) Lc[64 * q] = x[q] + p;
      }
    }
  }
  panel_rows(sh, pos, wrow, nw, kb, f.piv + s.ro + kb, mv);
}

// One wavefront per front of up to 64 rows: the front and its right-hand
// side (column m) in LDS, where the children's contribution blocks are added
// in child order, then in registers as 16 x 16 tiles, factored like a panel
// above (four columns at a time to a row per lane, rank-4 matrix-core
// products of the rest), every column at once.  Same operations per element
// as the other forms, so the same bits.  A front is a chain of column steps
// of ~0.5 us; with 16-column panels in LDS and separate passes for swaps, U12
// and update, 100 x 100 power-grid levels took 62 us on average.
template <int kNT, int kCT>
__global__ void __launch_bounds__(64) front_wave_kernel(FrontArgs f, int lv0) {
  __shared__ double F[16 * kNT][16 * kCT + 1];
  __shared__ __align__(16) double S[16 * kNT][4], srow[4][4];
  __shared__ double raw[4][16 * kCT];
  const int s = f.lv[lv0 + blockIdx.x];
  const int comp = f.comp[s];
  if (__builtin_amdgcn_readfirstlane(front_skip(f, comp))) return;  // one value for all lanes
  const int m = f.m[s], k = f.k[s];
  if (m > f.big_m) return;  // factored by many workgroups
  const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
  double *A = f.vals + f.fo[s], *w = f.wrhs + f.ro[s];
  auto fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const int row = min(lane, m - 1);
#pragma unroll 8
  for (int i = 0; i < m; ++i) {
    const double v = A[i * m + row];
    if (lane < m) F[i][lane] = v;
  }
  if (lane < m) F[lane][m] = w[lane];
  fence();
  // the children, their numbers a lane each (a merged front has dozens), and
  // each child's map, right-hand side and first kAhead rows read while the
  // one before it is added (one after the other they cost ~1.5 us each)
  constexpr int kAhead = 8;
  struct Child {
    int wc, mc, map;
    const double *C;
    double r, v[kAhead];
  };
  const int ch1 = f.ch_ptr[s + 1];
  for (int b = f.ch_ptr[s]; b < ch1; b += 64) {
    const int nb = min(64, ch1 - b);
    const int ch = f.ch[min(b + lane, ch1 - 1)];
    const int cm = f.m[ch], ck = f.k[ch];
    const int64_t cf = f.fo[ch] + (int64_t)ck * cm + ck, cr = f.ro[ch] + ck;
    auto fetch = [&](int q, Child &c) {
      auto word = [&](int v) { return __builtin_amdgcn_readlane(v, q); };
      auto wide = [&](int64_t v) {
        return (int64_t)(uint32_t)word((int)v) | (int64_t)word((int)(v >> 32)) << 32;
      };
      c.mc = word(cm);
      c.wc = c.mc - word(ck);
      c.C = f.vals + (c.wc > 0 ? wide(cf) : 0);
      const int jl = min(lane, max(c.wc - 1, 0));
      const int64_t ro = c.wc > 0 ? wide(cr) + jl : 0;
      c.map = f.cbmap[ro];
      c.r = f.wrhs[ro];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) c.v[i] = c.C[min(i, max(c.wc - 1, 0)) * c.mc + jl];
    };
    Child cur, nxt;
    fetch(0, cur);
    for (int q = 0; q < nb; ++q) {
      fetch(min(q + 1, nb - 1), nxt);
      const bool on = lane < cur.wc;
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int mi = __builtin_amdgcn_readlane(cur.map, i);
        if (on && i < cur.wc) F[mi][cur.map] += cur.v[i];
      }
#pragma unroll 8
      for (int i = kAhead; i < cur.wc; ++i) {
        const double v = cur.C[i * cur.mc + min(lane, cur.wc - 1)];
        const int mi = __builtin_amdgcn_readlane(cur.map, i);
        if (on) F[mi][cur.map] += v;
      }
      if (on) F[cur.map][m] += cur.r;
      fence();
      cur = nxt;
    }
  }
  double4v acc[kNT][kCT];
#pragma unroll
  for (int t = 0; t < kNT; ++t)
#pragma unroll
    for (int c = 0; c < kCT; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][c][r] = F[16 * t + lk + 4 * r][16 * c + li];
  int pos = lane < k ? lane : lane < m ? lane + 64 : -1;  // (rows >= k: no candidates)
#pragma unroll 1
  for (int c0 = 0; c0 < k; c0 += 4) {
    const int ct = c0 >> 4, nv = min(4, k - c0);
#pragma unroll
    for (int q = 0; q < kCT; ++q)
      if (ct == q) {
        if ((li >> 2) == ((c0 >> 2) & 3))
#pragma unroll
          for (int t = 0; t < kNT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[16 * t + lk + 4 * r][li & 3] = acc[t][q][r];
        asm volatile("; tile %0" ::"n"(q));  // (kept apart: fixed registers)
      }
    fence();
    double a[4], ln[4];
    const int sr = min(lane, 16 * kNT - 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[j] = S[sr][j];
      ln[j] = -0.0;
    }
    unsigned win = 0;  // the rows of the four pivots, eight bits each
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = c0 + j;
      if (j >= nv) continue;
      const bool cand = pos >= c && pos < k;
      const double v = cand ? fabs(a[j]) : 0.0;
      double rcp = make_pivot(a[j]).r;
      // (a NaN is no candidate, as in the other forms)
      const int wl = lane_of_max<6>(v > 0.0 ? v : 0.0, cand ? pos : 0x7fffffff);
      const double best = read_lane(v, wl);
      const int bp = __builtin_amdgcn_readlane(pos, wl);
      rcp = read_lane(rcp, wl);
      if (!(best > 0.0) || !(best <= DBL_MAX)) {  // the same in every lane
        if (lane == 0) f.bad[comp] = 1;
        return;
      }
      win |= (unsigned)wl << (8 * j);
      if (lane == wl)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) srow[j][jj] = a[jj];
      fence();
      double u[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) u[jj] = srow[j][jj];
      if (lane >= j && lane < nv) A[c * m + c0 + lane] = srow[j][lane];
      const Pivot pv{__builtin_amdgcn_frexp_mant(u[j]), rcp, -__builtin_amdgcn_frexp_exp(u[j])};
      pos = pos == bp ? c : (pos == c ? bp : pos);
      if (pos > c) {
        const double l = divide(a[j], pv);
        a[j] = l;
        ln[j] = -l;
#pragma unroll
        for (int jj = j + 1; jj < 4; ++jj) a[jj] = fma(-l, u[jj], a[jj]);
      }
    }
    // the pivot rows' other columns, from the lanes that hold them
#pragma unroll 1
    for (int j = 0; j < nv; ++j) {
      const int ph = win >> (8 * j) & 255;
#pragma unroll
      for (int t = 0; t < kNT; ++t)
        if ((ph >> 4) == t) {
          const int r = (ph >> 2) & 3;
#pragma unroll
          for (int q = 0; q < kCT; ++q) {
            const double4v x = acc[t][q];
            const double y = r == 0 ? x[0] : r == 1 ? x[1] : r == 2 ? x[2] : x[3];
            if (lk == (ph & 3)) raw[j][16 * q + li] = y;
          }
          asm volatile("; tile %0" ::"n"(t));
        }
    }
    if (lane < 16 * kNT)
#pragma unroll
      for (int j = 0; j < 4; ++j) S[lane][j] = ln[j];
    fence();
    double av[kNT];
#pragma unroll
    for (int t = 0; t < kNT; ++t) av[t] = S[16 * t + li][lk];
    double l[4][4];
#pragma unroll
    for (int j = 1; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < j; ++i) l[j][i] = srow[j][i];
#pragma unroll
    for (int q = 0; q < kCT; ++q) {
      if (q < ct) continue;
      double u[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u[j] = raw[j][16 * q + li];
#pragma unroll
        for (int i = 0; i < j; ++i) u[j] = fma(-l[j][i], u[i], u[j]);
      }
      const int col = 16 * q + li;
      const double x = lk == 0 ? u[0] : lk == 1 ? u[1] : lk == 2 ? u[2] : u[3];
      const bool on = col >= c0 + nv && lk < nv;
      if (on && col < m) A[(c0 + lk) * m + col] = x;
      if (on && col == m) w[c0 + lk] = x;
      const double ub = on ? x : 0.0;
#pragma unroll
      for (int t = 0; t < kNT; ++t)
        acc[t][q] = add_group(av[t], ub, acc[t][q]);
    }
    fence();
  }
  // the contribution block and its right-hand side
#pragma unroll
  for (int t = 0; t < kNT; ++t)
#pragma unroll
    for (int c = 0; c < kCT; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * t + lk + 4 * r, j = 16 * c + li;
        if (i >= k && i < m && j >= k && j < m) A[i * m + j] = acc[t][c][r];
        if (i >= k && i < m && j == m) w[i] = acc[t][c][r];
      }
}

// After a panel.  Workgroups [0, column blocks): a lane per column j >= cl
// (j = m the right-hand side): the rows the swaps bring into the panel's
// block and the block's rows they displace, all loaded at once, then U12 =
// L11^-1 (by groups of four pivots).  The others: a lane
// per row >= k, L21 = A21 U11^-1 through a transposing LDS tile (each entry
// updated group by group, then divided by its pivot, as the
// right-looking form does), to the panel buffer.  One swap at a time, each
// waiting for the last one's stores, took 40 us per panel of the 5,000-gate
// logic.
__global__ void __launch_bounds__(64) front_solve_kernel(FrontArgs f, int lb, int kb, int wp) {
  __shared__ double D[kBigW][kBigW + 1];
  __shared__ double T[64][kBigW + 1];
  __shared__ double dr[kBigW];
  __shared__ int32_t top[kBigW], mdst[kBigW], msrc[kBigW];
  const BigFront s = f.big[lb + blockIdx.y];
  // (another front's workgroup may set the flag just now; either value will do,
  // and this workgroup is one wavefront)
  if (__builtin_amdgcn_readfirstlane(front_skip(f, s.comp))) return;
  const int m = s.m, k = s.k;
  if (kb >= k) return;
  const int cl = min(kb + wp, k), nw = cl - kb;
  const int ncb = (m + 1 - cl + 63) / 64, nrb = (m - k + 63) / 64;
  const int lane = threadIdx.x;
  const int b = blockIdx.x;
  if (b >= ncb + nrb) return;
  double *A = f.vals + s.fo;
  double *L = f.lbuf + s.lo;
  constexpr int RI = 64 / kBigW;
  const int lr = lane / kBigW, lc = lane % kBigW;
  if (b < ncb) {
    const int32_t *mv = f.mv + (int64_t)blockIdx.y * kMoveInts;
    const int nm = mv[0];
    if (nm < 0) {  // the panel found no pivot: no rows and no multipliers of it
      if (b == 0 && lane == 0) f.bad[s.comp] = 1;
      return;
    }
    if (lane < kBigW) {  // (padded with readable rows, so no load below is conditional)
      top[lane] = lane < nw ? f.piv[s.ro + kb + lane] : kb;
      mdst[lane] = lane < nm ? mv[1 + 2 * lane] : kb;
      msrc[lane] = lane < nm ? mv[2 + 2 * lane] : kb;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kBigW / RI; ++i) {  // L11, columns in rows of D
      const int c = i * RI + lr;
      D[c][lc] = load_if((c < lc) & (lc < nw), L, (int64_t)c * m + top[lc]);
    }
    const int j = cl + b * 64 + lane, jc = min(j, m);
    double *col = jc < m ? A + jc : f.wrhs + s.ro;
    const int ld = jc < m ? m : 1;
    double u[kBigW], d[kBigW];
#pragma unroll
    for (int c = 0; c < kBigW; ++c) u[c] = col[top[c] * ld];
#pragma unroll
    for (int c = 0; c < kBigW; ++c) d[c] = col[msrc[c] * ld];
#pragma unroll
    for (int c = 0; c < kBigW; ++c) asm("" : "+v"(d[c]));  // (not sunk to their stores)
    __syncthreads();
    if (j > m) return;
#pragma unroll
    for (int c = 0; c < kBigW; ++c)
      if (c < nm) col[mdst[c] * ld] = d[c];
#pragma unroll
    for (int g = 0; g < kBigW; g += 4) {
#pragma unroll
      for (int c = g; c < g + 4; ++c)
        if (c < nw)
#pragma unroll
          for (int i = c + 1; i < g + 4; ++i) u[i] = fma(-D[c][i], u[c], u[i]);
      if (g + 4 < nw)  // (a group with rows after it is whole)
#pragma unroll
        for (int i = g + 4; i < kBigW; ++i) {
          double p = 0.0;
#pragma unroll
          for (int c = g; c < g + 4; ++c) p = fma(-D[c][i], u[c], p);
          u[i] = u[i] + p;
        }
      __builtin_amdgcn_sched_barrier(0);  // D's reads stay by their group
    }
#pragma unroll
    for (int c = 0; c < kBigW; ++c)
      if (c < nw) col[(kb + c) * ld] = u[c];
    return;
  }
#pragma unroll
  for (int i = 0; i < kBigW / RI; ++i) {
    const int r = i * RI + lr;
    D[r][lc] = load_if((r <= lc) & (lc < nw), A, (int64_t)(kb + r) * m + kb + lc);
  }
  const int r0 = k + (b - ncb) * 64;
#pragma unroll
  for (int i = 0; i < 64 / RI; ++i) {
    const int r = min(r0 + i * RI + lr, m - 1);
    T[i * RI + lr][lc] = A[(int64_t)r * m + kb + min(lc, nw - 1)];
  }
  __syncthreads();
  if (lane < kBigW) dr[lane] = make_pivot(D[lane][lane]).r;
  __syncthreads();
  double l[kBigW];
#pragma unroll
  for (int c = 0; c < kBigW; ++c) l[c] = T[lane][c];
#pragma unroll
  for (int g = 0; g < kBigW; g += 4) {
#pragma unroll
    for (int c = g; c < g + 4; ++c)
      if (c < nw) {
        const double d = D[c][c];
        l[c] = divide(l[c], {__builtin_amdgcn_frexp_mant(d), dr[c], -__builtin_amdgcn_frexp_exp(d)});
#pragma unroll
        for (int i = c + 1; i < g + 4; ++i) l[i] = fma(-l[c], D[c][i], l[i]);
        if (r0 + lane < m) L[(int64_t)c * m + r0 + lane] = l[c];
      }
    if (g + 4 < nw)
#pragma unroll
      for (int i = g + 4; i < kBigW; ++i) {
        double p = 0.0;
#pragma unroll
        for (int c = g; c < g + 4; ++c) p = fma(-l[c], D[c][i], p);
        l[i] = l[i] + p;
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Rows and columns >= cl: A -= L21 U12, and the right-hand side's rows.
// Grid: (tiles over columns, tiles over rows, fronts).  Each wavefront takes
// a 32 x 32 quarter of the tile as 2 x 2 products of 16 x 16 x 4
// (v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// D[l / 16 + 4 r][l % 16]; its result is the fused multiply-adds in
// ascending k, so these are the bits of the scalar form).  One element per
// thread with two LDS reads per multiply-add took 21 us per panel of the
// 5,000-gate logic.
__global__ void __launch_bounds__(kFB) front_update_kernel(FrontArgs f, int lb, int kb,
                                                           int wp) {
  __shared__ double Lt[kBigW][kTile + 1];  // -L21, columns in rows
  __shared__ double Ut[kBigW][kTile + 1];
  __shared__ double y[kBigW];
  const BigFront s = f.big[lb + blockIdx.z];
  if (front_skip(f, s.comp)) return;
  const int m = s.m, k = s.k;
  if (kb >= k) return;
  const int cl = min(kb + wp, k), nw = cl - kb;
  double *A = f.vals + s.fo, *w = f.wrhs + s.ro;
  const int r0 = cl + blockIdx.y * kTile, c0 = cl + blockIdx.x * kTile;
  if (r0 >= m || c0 >= m) return;
  const int t = threadIdx.x;
  const int wave = t >> 6, lane = t & 63, li = lane & 15, lk = lane >> 4;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  double4v acc[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = r0 + wr + 16 * p + lk + 4 * r, j = c0 + wc + 16 * q + li;
        acc[p][q][r] = load_if((i < m) & (j < m), A, (int64_t)i * m + j);
      }
  // padding: a product of -0.0, the identity of the sum
  {
    // (rows below the fully summed block stay where they are)
    const int i = r0 + lane;
    const int src = i < k ? f.piv[s.ro + i] : i;
    const double *L = f.lbuf + s.lo;
#pragma unroll
    for (int q = 0; q < kBigW / 4; ++q) {
      const int cc = 4 * q + wave;
      Lt[cc][lane] = -load_if((i < m) & (cc < nw), L, (int64_t)cc * m + src);
    }
  }
#pragma unroll
  for (int e = t; e < kBigW * kTile; e += kFB) {
    const int cc = e / kTile, q = e % kTile;
    Ut[cc][q] = load_if((cc < nw) & (c0 + q < m), A, (int64_t)(kb + cc) * m + c0 + q);
  }
  if (t < kBigW) y[t] = t < nw ? w[kb + t] : 0.0;
  __syncthreads();
  for (int kk = 0; kk < nw; kk += 4) {
    double av[2], bv[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      av[p] = Lt[kk + lk][wr + 16 * p + li];
      bv[p] = Ut[kk + lk][wc + 16 * p + li];
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        acc[p][q] = add_group(av[p], bv[q], acc[p][q]);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = r0 + wr + 16 * p + lk + 4 * r, j = c0 + wc + 16 * q + li;
        if (i < m && j < m) A[(int64_t)i * m + j] = acc[p][q][r];
      }
  if (blockIdx.x == 0 && t < kTile && r0 + t < m) {
    double v = w[r0 + t];
    for (int g = 0; g < nw; g += 4) {  // (padded like the tiles)
      double p = 0.0;
#pragma unroll
      for (int cc = g; cc < g + 4; ++cc) p = fma(Lt[cc][t], y[cc], p);
      v = v + p;
    }
    w[r0 + t] = v;
  }
}

// Backward solve of one level's fronts (levels from the root down): the
// rows below the fully summed block are solved already (by ancestors).
// First the right-hand side less the solved rows below, a wavefront per
// row: lane-strided products, summed by wave_sum.  Then blocks of 64 columns
// from the last: the diagonal block in LDS on the first wavefront, a lane
// per row, while the others subtract the block solved before it from the
// rows above (the rows of the next block first, by everyone), eight lanes a
// row.  The chain of the diagonal blocks (~100 cycles a column: the
// quotient, its broadcast, the update) and one CU's reads of U are about
// equal for the largest fronts; with a row per thread and the diagonal read
// from memory inside the chain a 1540-row front took 1 ms.
template <int ROWS, int BS>
__global__ void __launch_bounds__(BS) front_bwd_kernel(FrontArgs f, int lv0) {
  constexpr int NW = BS / 64;
  __shared__ double tb[ROWS], xs[ROWS], D[64][65];
  const int s = f.lv[lv0 + blockIdx.x];
  const int c = f.comp[s];
  if (front_skip(f, c)) return;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int m = f.m[s], k = f.k[s];
  const double *A = f.vals + f.fo[s];
  const int32_t *rows = f.rows + f.ro[s];
  const double *y = f.wrhs + f.ro[s];
  for (int j = k + t; j < m; j += BS) xs[j - k] = f.v[rows[j]];
  __syncthreads();
  for (int i = w; i < k; i += NW) {
    const double *a = A + (int64_t)i * m;
    double p = 0.0;
#pragma unroll 4
    for (int j = k + lane; j < m; j += 64) p = fma(a[j], xs[j - k], p);
    p = wave_sum(p);
    if (lane == 0) tb[i] = y[i] - p;
  }
  // rows [r0, r1) less their columns [c0, c1) times the solved tb there, by
  // nt threads of which this one is `id`
  auto subtract = [&](int r0, int r1, int c0, int c1, int id, int nt) {
    const int sub = id & 7;
    double x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = load_if(c0 + 8 * sub + q < c1, tb, c0 + 8 * sub + q);
#pragma unroll 2
    for (int r = r0 + (id >> 3); r < r1; r += nt / 8) {
      const double *a = A + (int64_t)r * m;
      double v[8], p = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = load_if(c0 + 8 * sub + q < c1, a, c0 + 8 * sub + q);
#pragma unroll
      for (int q = 0; q < 8; ++q) p = fma(v[q], x[q], p);
      p = sum8(p);
      if (sub == 0) tb[r] = tb[r] - p;
    }
  };
  for (int jb = ((k - 1) / 64) * 64; jb >= 0; jb -= 64) {
    const int je = min(jb + 64, k), n = je - jb, je2 = min(je + 64, k);
    double d[64 * 64 / BS];
#pragma unroll
    for (int q = 0; q < 64 * 64 / BS; ++q) {
      const int e = t + q * BS, r = e >> 6, cc = e & 63;
      d[q] = load_if((r <= cc) & (cc < n), A, (int64_t)(jb + r) * m + jb + cc);
    }
    __syncthreads();  // tb of the block before, and D free
    if (je < k) subtract(jb, je, je, je2, t, BS);
#pragma unroll
    for (int q = 0; q < 64 * 64 / BS; ++q) {
      const int e = t + q * BS;
      D[e >> 6][e & 63] = d[q];
    }
    __syncthreads();
    if (w == 0) {
      double ti = load_if(lane < n, tb, jb + lane);
      const Pivot pv = make_pivot(lane < n ? D[lane][lane] : 1.0);
      double dj = D[lane][n - 1];
      for (int j = n - 1; j >= 0; --j) {
        const double dn = D[lane][max(j - 1, 0)];
        const double xj = read_lane(divide(ti, pv), j);
        ti = lane < j ? fma(-dj, xj, ti) : lane == j ? xj : ti;
        dj = dn;
      }
      if (lane < n) tb[jb + lane] = ti;
    } else if (je < k) {
      subtract(0, jb, je, je2, t - 64, BS - 64);
    }
  }
  __syncthreads();
  for (int i = t; i < k; i += BS) f.v[rows[i]] = tb[i];
}

// The same for fronts of up to kTinyM rows, one thread each, with the same
// operations per element (the products summed as wave_sum sums them).
__global__ void __launch_bounds__(64) front_tiny_bwd_kernel(FrontArgs f, int lv0, int nfr) {
  const int q = blockIdx.x * 64 + threadIdx.x;
  if (q >= nfr) return;
  const int s = f.lv[lv0 + q];
  const int c = f.comp[s];
  if (front_skip(f, c)) return;
  const int m = f.m[s], k = f.k[s];
  const double *A = f.vals + f.fo[s];
  const int32_t *rows = f.rows + f.ro[s];
  double *y = f.wrhs + f.ro[s];
  double x[kTinyM];
#pragma unroll
  for (int j = 0; j < kTinyM; ++j) x[j] = load_if(k + j < m, f.v, rows[min(k + j, m - 1)]);
  for (int i = 0; i < k; ++i) {
    double p[kTinyM];
#pragma unroll
    for (int j = 0; j < kTinyM; ++j) p[j] = fma(load_if(k + j < m, A, i * m + k + j), x[j], 0.0);
#pragma unroll
    for (int st = 1; st < kTinyM; st *= 2)
#pragma unroll
      for (int j = 0; j < kTinyM; j += 2 * st) p[j] = p[j] + p[j + st];
    // (wave_sum's empty lanes: at least one zero more in every step)
    y[i] = y[i] - (((p[0] + 0.0) + 0.0) + 0.0);
  }
  for (int j = k - 1; j >= 0; --j) {
    const double xj = divide(y[j], make_pivot(A[j * m + j]));
    f.v[rows[j]] = xj;
    for (int i = 0; i < j; ++i) y[i] = fma(-A[i * m + j], xj, y[i]);
  }
}

// The residual and |J| row-sum maxima of a component's long rows in
// [r0, r1) (rows of more than kLongRow entries, listed per component):
// each row by the whole block, strided partial sums then a fixed tree.
template <int B>
__device__ void long_rows_check(const FrontArgs &f, const SparseLuArgs &a, int c, int r0,
                                int r1, double *sv, double &rm, double &am) {
  const int beg = a.cstart[c];
  const int eb = a.ent_off[c];
  const double *jp = a.Jp + eb;
  const int32_t *ecol = a.ent_col + eb, *ers = a.ent_rs + beg + c;
  const double *v = f.v + beg;
  for (int q = f.long_ptr[c]; q < f.long_ptr[c + 1]; ++q) {
    const int i = f.long_rows[q];
    if (i < r0 || i >= r1) continue;
    double s = 0.0, as = 0.0;
    for (int j = ers[i] + threadIdx.x; j < ers[i + 1]; j += B) {
      const double qv = jp[j];
      s = s + qv * v[ecol[j]];
      as = as + fabs(qv);
    }
    s = blk_reduce<B>(s, sv, false);
    as = blk_reduce<B>(as, sv, false);
    rm = fmax(rm, fabs(a.bp[beg + i] - s));
    am = fmax(am, as);
  }
}

// Per front component: backward error of the solution against the
// unfactored rows (entry-ordered J and position-ordered rhs of the permute
// kernel), then x += dx and the weighted RMS norm of dx
// (N_NLS_DampedNewton.C:311-335), as the task-list kernel does.
__global__ void __launch_bounds__(kFinishBlock) front_finish_kernel(FrontArgs f,
                                                                    SparseLuArgs a) {
  __shared__ double sv[kFinishBlock];
  const int c = blockIdx.x;
  const int t = threadIdx.x;
  if (f.gate && *f.gate) return;
  if (!f.front_comp[c]) return;
  if (f.fin_split && f.fin_split[c]) return;  // the chunked kernels below
  if (a.active && !a.active[c]) return;  // stats written by the task kernel
  const int beg = a.cstart[c], n = a.cstart[c + 1] - beg;
  double *stats = a.stats + 4 * (size_t)c;
  double rmax = 0.0;
  for (int i = t; i < n; i += kFinishBlock) rmax = fmax(rmax, fabs(a.bp[beg + i]));
  const double max_rhs = blk_reduce<kFinishBlock>(rmax, sv, true);
  bool good = !f.bad[c];
  if (good) {
    const int eb = a.ent_off[c];
    const double *jp = a.Jp + eb;
    const int32_t *ecol = a.ent_col + eb, *ers = a.ent_rs + beg + c;
    const double *v = f.v + beg;
    double rm = 0.0, am = 0.0, xm = 0.0;
    for (int i = t; i < n; i += kFinishBlock) {
      xm = fmax(xm, fabs(v[i]));
      if (ers[i + 1] - ers[i] > kLongRow) continue;  // below, by the block
      double r = a.bp[beg + i], as = 0.0;
      for (int j = ers[i]; j < ers[i + 1]; ++j) {
        const double q = jp[j];
        r = r - q * v[ecol[j]];
        as = as + fabs(q);
      }
      rm = fmax(rm, fabs(r));
      am = fmax(am, as);
    }
    long_rows_check<kFinishBlock>(f, a, c, 0, n, sv, rm, am);
    rm = blk_reduce<kFinishBlock>(rm, sv, true);
    am = blk_reduce<kFinishBlock>(am, sv, true);
    xm = blk_reduce<kFinishBlock>(xm, sv, true);
    good = rm <= a.max_berr * (am * xm + max_rhs);  // false for NaN / inf too
  }
  if (!good) {
    // singular for the fronts' restricted pivoting: the dense partial-
    // pivoting kernel launched next refactors the component when it has a
    // dense form, and reports it singular otherwise
    if (t == 0) {
      stats[0] = max_rhs;
      stats[1] = 0.0;
      stats[2] = 1.0;
      stats[3] = (double)n;
      a.fallback[c] = 1;
    }
    return;
  }
  const int32_t *qcol = a.qcol + beg;
  double acc = 0.0;
  for (int i = t; i < n; i += kFinishBlock) {
    const int g = qcol[i];
    const double dx = f.v[beg + i];
    const double w = a.reltol * fmax(fabs(a.wa[g]), fabs(a.wb[g])) + a.abstol;
    const double q = dx / w;
    acc = acc + q * q;
    a.x[g] = a.x[g] + dx;
  }
  const double ss = blk_reduce<kFinishBlock>(acc, sv, false);
  if (t == 0) {
    stats[0] = max_rhs;
    stats[1] = sqrt(ss / n);
    stats[2] = 0.0;
    stats[3] = (double)n;
  }
}

// ---- the same finish for components of more than kFinishSplit unknowns,
// in chunks of kFinishChunk rows: (1) per chunk the maxima of |rhs|, of
// the residual, of the row sums of |J| and of |dx|; (2) per component
// their maxima (exact in any order) and the verdict; (3) per chunk
// x += dx and the chunk's sum of squared weighted steps; (4) per component
// those sums in chunk order, the weighted RMS norm.
__global__ void __launch_bounds__(kFB) finish_part_kernel(FrontArgs f, SparseLuArgs a) {
  __shared__ double sv[kFB];
  if (f.gate && *f.gate) return;
  const int ch = blockIdx.x, t = threadIdx.x;
  const int c = f.fin_chunk_comp[ch];
  if (a.active && !a.active[c]) return;
  const int beg = a.cstart[c], n = a.cstart[c + 1] - beg;
  const int r0 = f.fin_chunk_beg[ch], r1 = min(n, r0 + kFinishChunk);
  double rmax = 0.0, rm = 0.0, am = 0.0, xm = 0.0;
  const bool bad = f.bad[c] != 0;
  const int eb = a.ent_off[c];
  const double *jp = a.Jp + eb;
  const int32_t *ecol = a.ent_col + eb, *ers = a.ent_rs + beg + c;
  const double *v = f.v + beg;
  for (int i = r0 + t; i < r1; i += kFB) {
    const double b = a.bp[beg + i];
    rmax = fmax(rmax, fabs(b));
    if (!bad) {
      xm = fmax(xm, fabs(v[i]));
      if (ers[i + 1] - ers[i] > kLongRow) continue;  // below, by the block
      double r = b, as = 0.0;
      for (int j = ers[i]; j < ers[i + 1]; ++j) {
        const double q = jp[j];
        r = r - q * v[ecol[j]];
        as = as + fabs(q);
      }
      rm = fmax(rm, fabs(r));
      am = fmax(am, as);
    }
  }
  if (!bad) long_rows_check<kFB>(f, a, c, r0, r1, sv, rm, am);
  double *p = f.fin_part + 4 * (size_t)ch;
  rmax = blk_reduce<kFB>(rmax, sv, true);
  rm = blk_reduce<kFB>(rm, sv, true);
  am = blk_reduce<kFB>(am, sv, true);
  xm = blk_reduce<kFB>(xm, sv, true);
  if (t == 0) {
    p[0] = rmax;
    p[1] = rm;
    p[2] = am;
    p[3] = xm;
  }
}

__global__ void __launch_bounds__(kFB) finish_decide_kernel(FrontArgs f, SparseLuArgs a) {
  __shared__ double sv[kFB];
  if (f.gate && *f.gate) return;
  const int c = f.fin_comps[blockIdx.x], t = threadIdx.x;
  if (a.active && !a.active[c]) return;
  const int n = a.cstart[c + 1] - a.cstart[c];
  double m4[4] = {0.0, 0.0, 0.0, 0.0};
  for (int ch = f.fin_cptr[blockIdx.x] + t; ch < f.fin_cptr[blockIdx.x + 1]; ch += kFB)
    for (int q = 0; q < 4; ++q) m4[q] = fmax(m4[q], f.fin_part[4 * (size_t)ch + q]);
  for (int q = 0; q < 4; ++q) m4[q] = blk_reduce<kFB>(m4[q], sv, true);
  const bool good = !f.bad[c] && m4[1] <= a.max_berr * (m4[2] * m4[3] + m4[0]);
  if (t == 0) {
    f.fin_good[c] = good ? 1 : 0;
    double *stats = a.stats + 4 * (size_t)c;
    stats[0] = m4[0];
    if (!good) {
      stats[1] = 0.0;
      stats[2] = 1.0;
      stats[3] = (double)n;
      a.fallback[c] = 1;
    }
  }
}

__global__ void __launch_bounds__(kFB) finish_update_kernel(FrontArgs f, SparseLuArgs a) {
  __shared__ double sv[kFB];
  if (f.gate && *f.gate) return;
  const int ch = blockIdx.x, t = threadIdx.x;
  const int c = f.fin_chunk_comp[ch];
  if (a.active && !a.active[c]) return;
  if (!f.fin_good[c]) return;
  const int beg = a.cstart[c], n = a.cstart[c + 1] - beg;
  const int r0 = f.fin_chunk_beg[ch], r1 = min(n, r0 + kFinishChunk);
  const int32_t *qcol = a.qcol + beg;
  double acc = 0.0;
  for (int i = r0 + t; i < r1; i += kFB) {
    const int g = qcol[i];
    const double dx = f.v[beg + i];
    const double w = a.reltol * fmax(fabs(a.wa[g]), fabs(a.wb[g])) + a.abstol;
    const double q = dx / w;
    acc = acc + q * q;
    a.x[g] = a.x[g] + dx;
  }
  acc = blk_reduce<kFB>(acc, sv, false);
  if (t == 0) f.fin_part[4 * (size_t)ch] = acc;
}

__global__ void __launch_bounds__(64) finish_sum_kernel(FrontArgs f, SparseLuArgs a) {
  if (f.gate && *f.gate) return;
  const int c = f.fin_comps[blockIdx.x];
  if (a.active && !a.active[c]) return;
  if (!f.fin_good[c] || threadIdx.x != 0) return;
  const int n = a.cstart[c + 1] - a.cstart[c];
  double ss = 0.0;
  for (int ch = f.fin_cptr[blockIdx.x]; ch < f.fin_cptr[blockIdx.x + 1]; ++ch)
    ss = ss + f.fin_part[4 * (size_t)ch];
  double *stats = a.stats + 4 * (size_t)c;
  stats[1] = sqrt(ss / n);
  stats[2] = 0.0;
  stats[3] = (double)n;
}

// Most fronts of up to 64 rows in a level for each to take a wavefront, the
// ones of up to kTinyM rows included (in place of a launch of their own, a
// thread each).
constexpr int kWaveFronts = 2048;

// One workgroup per front of the level (fronts above 64 rows, when the
// many-workgroup threshold is raised).
template <int NB, int ROWS>
hipError_t launch_level(const FrontArgs &f, int lv0, int nfr, hipStream_t s) {
  hipLaunchKernelGGL((front_factor_kernel<NB, ROWS, kFB>), dim3(nfr), dim3(kFB), 0, s, f, lv0);
  return hipGetLastError();
}

// The panel launch for `nr` fully summed rows left, its width: 32 columns
// while a lane holds at most two rows, so that the tiles fit the registers of
// eight wavefronts (256 a lane), 16 above; from 2048 rows on they wait in
// memory.
int launch_panel(const FrontArgs &f, int lb, int nb, int kb, int nr, hipStream_t s) {
#define XG_PANEL(NW, NT, CT)                                                             \
  do {                                                                                   \
    hipLaunchKernelGGL((front_panel_kernel<NW, NT, CT>), dim3(nb), dim3(64 * NW), 0, s, f, \
                       lb, kb);                                                          \
    return 16 * CT;                                                                      \
  } while (0)
  if (nr <= 64) XG_PANEL(1, 4, 2);
  if (nr <= 256) XG_PANEL(4, 4, 2);
  if (nr <= 512) XG_PANEL(8, 4, 2);
  if (nr <= 1024) XG_PANEL(8, 8, 2);
  if (nr <= 2048) XG_PANEL(8, 16, 1);
#undef XG_PANEL
  hipLaunchKernelGGL((front_tall_panel_kernel<8, 7>), dim3(nb), dim3(64 * 8), 0, s, f, lb, kb);
  return 16;
}

// A level's fronts of more than big_m rows (f.big[lb, lb + nb)) by many
// workgroups: their children's contribution blocks (one launch, a
// workgroup per receiving row), then per panel position the panel, solve
// and trailing-update launches over all of them.
hipError_t launch_big_fronts(const FrontArgs &f, int lb, int nb, hipStream_t s) {
  int max_k = 0;
  int64_t max_rows = 0;
  for (int q = lb; q < lb + nb; ++q) {
    const BigFront &b = f.big_host[q];
    max_k = std::max(max_k, b.k);
    max_rows = std::max(max_rows, b.xr1 - b.xr0);
  }
  if (max_rows > 0)
    hipLaunchKernelGGL(front_extend_kernel, dim3((unsigned)max_rows, nb), dim3(kFB), 0, s, f,
                       lb);
  for (int kb = 0; kb < max_k;) {
    const int wp = launch_panel(f, lb, nb, kb, max_k - kb, s);
    // the largest trailing block and solve at this panel position
    int rest = 0, blocks = 0;
    for (int q = lb; q < lb + nb; ++q) {
      const int m = f.big_host[q].m, k = f.big_host[q].k;
      if (kb >= k) continue;
      const int r = m - std::min(kb + wp, k);
      rest = std::max(rest, r);
      blocks = std::max(blocks, (r + 1 + 63) / 64 + (m - k + 63) / 64);
    }
    hipLaunchKernelGGL(front_solve_kernel, dim3(blocks, nb), dim3(64), 0, s, f, lb, kb, wp);
    if (rest > 0) {
      const unsigned tiles = (unsigned)((rest + kTile - 1) / kTile);
      hipLaunchKernelGGL(front_update_kernel, dim3(tiles, tiles, nb), dim3(kFB), 0, s, f, lb,
                         kb, wp);
    }
    kb += wp;
  }
  return hipGetLastError();
}

}  // namespace

// The panel form for fronts of up to `max_m` rows: 0 when none fits.
int front_form(int32_t max_m) {
  if (max_m <= 64) return 1;
  if (max_m <= 256) return 2;
  if (max_m <= 1024) return 3;
  if (max_m <= 1934) return 4;
  if (max_m <= kFrontMaxM) return 5;
  return 0;
}

hipError_t launch_fronts(const FrontArgs &f, const SparseLuArgs &a, hipStream_t s) {
  if (f.n_fronts == 0) return hipSuccess;
  const unsigned gclear =
      (unsigned)std::min<int64_t>((std::max(f.n_vals, (int64_t)f.n_comp) + kFB - 1) / kFB, 8192);
  hipLaunchKernelGGL(front_clear_kernel, dim3(gclear), dim3(kFB), 0, s, f, a.bp);
  const unsigned gsc = (unsigned)std::min<int64_t>((f.n_ent + kFB - 1) / kFB + 1, 8192);
  hipLaunchKernelGGL(front_scatter_kernel, dim3(gsc), dim3(kFB), 0, s, f, a.J);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  for (int L = 0; L < f.n_levels; ++L) {
    // the level's fronts by size class (kTinyM rows, 64 rows, larger): those
    // up to 64 rows by threads and wavefronts, larger ones up to big_m rows
    // (when that is raised) by a workgroup each, the rest by many
    const int32_t *cp = f.cls_host + 3 * L;
    const int lv0 = cp[0], mid0 = cp[1], big0 = cp[2], lv1 = cp[3];
    int32_t one_max = 0;  // largest of the last class up to big_m rows
    for (int q = big0; q < lv1; ++q)
      if (f.m_host[f.lv_host[q]] <= f.big_m)
        one_max = std::max(one_max, f.m_host[f.lv_host[q]]);
    // (a level of few fronts: a wavefront for each of those up to 64 rows)
    const int wave0 = big0 - lv0 <= kWaveFronts ? lv0 : mid0;
    if (wave0 > lv0)
      hipLaunchKernelGGL(front_tiny_kernel, dim3((wave0 - lv0 + 63) / 64), dim3(64), 0, s, f,
                         lv0, wave0 - lv0);
    if (big0 > wave0) {
      // (they are in order of size: a level of many takes a launch per tile
      // count, so that the small ones have the registers and LDS of theirs)
      for (int q0 = wave0; q0 < big0;) {
        int q1 = big0;
        int32_t mx = f.m_host[f.lv_host[big0 - 1]];
        if (big0 - wave0 > kWaveFronts) {
          mx = std::min(64, f.m_host[f.lv_host[q0]] / 16 * 16 + 15);
          q1 = q0 + 1;
          while (q1 < big0 && f.m_host[f.lv_host[q1]] <= mx) ++q1;
        }
#define XG_WAVE(NT, CT) \
  hipLaunchKernelGGL((front_wave_kernel<NT, CT>), dim3(q1 - q0), dim3(64), 0, s, f, q0)
        if (mx <= 15) XG_WAVE(1, 1);
        else if (mx <= 31) XG_WAVE(2, 2);
        else if (mx <= 47) XG_WAVE(3, 3);
        else if (mx <= 63) XG_WAVE(4, 4);
        else XG_WAVE(4, 5);
#undef XG_WAVE
        q0 = q1;
      }
    }
    if (one_max > 0) {
      const int nfr = lv1 - big0;
      switch (front_form(one_max)) {
        case 2: e = launch_level<16, 256>(f, big0, nfr, s); break;
        case 3: e = launch_level<16, 1024>(f, big0, nfr, s); break;
        case 4: e = launch_level<8, 1934>(f, big0, nfr, s); break;
        default: e = launch_level<4, kFrontMaxM>(f, big0, nfr, s); break;
      }
      if (e != hipSuccess) return e;
    }
    // the level's larger fronts, at most kBigLaunch per launch (grid y / z)
    for (int lb = f.big_ptr_host[L]; lb < f.big_ptr_host[L + 1]; lb += kBigLaunch)
      if ((e = launch_big_fronts(f, lb, std::min(kBigLaunch, f.big_ptr_host[L + 1] - lb), s)) !=
          hipSuccess)
        return e;
  }
  // the backward solve's LDS holds a front's rows: the level's largest front
  // picks the instance (the largest fronts with 512 threads)
  for (int L = f.n_levels - 1; L >= 0; --L) {
    const int32_t *cp = f.cls_host + 3 * L;
    const int mm = f.lv_maxm_host[L];
    const int wave0 = cp[2] - cp[0] <= kWaveFronts ? cp[0] : cp[1];
    if (wave0 > cp[0])
      hipLaunchKernelGGL(front_tiny_bwd_kernel, dim3((wave0 - cp[0] + 63) / 64), dim3(64), 0, s,
                         f, cp[0], wave0 - cp[0]);
    if (cp[2] > wave0)
      hipLaunchKernelGGL((front_bwd_kernel<64, kFB>), dim3(cp[2] - wave0), dim3(kFB), 0, s, f,
                         wave0);
    if (cp[3] > cp[2]) {
      if (mm <= 512)
        hipLaunchKernelGGL((front_bwd_kernel<512, kFB>), dim3(cp[3] - cp[2]), dim3(kFB), 0, s, f,
                           cp[2]);
      else
        hipLaunchKernelGGL((front_bwd_kernel<kFrontMaxM, kSolveBlock>), dim3(cp[3] - cp[2]),
                           dim3(kSolveBlock), 0, s, f, cp[2]);
    }
  }
  hipLaunchKernelGGL(front_finish_kernel, dim3(f.n_comp), dim3(kFinishBlock), 0, s, f, a);
  if (f.n_fin_chunks > 0) {
    hipLaunchKernelGGL(finish_part_kernel, dim3(f.n_fin_chunks), dim3(kFB), 0, s, f, a);
    hipLaunchKernelGGL(finish_decide_kernel, dim3(f.n_fin_comps), dim3(kFB), 0, s, f, a);
    hipLaunchKernelGGL(finish_update_kernel, dim3(f.n_fin_chunks), dim3(kFB), 0, s, f, a);
    hipLaunchKernelGGL(finish_sum_kernel, dim3(f.n_fin_comps), dim3(64), 0, s, f, a);
  }
  return hipGetLastError();
}

}  // namespace xg
