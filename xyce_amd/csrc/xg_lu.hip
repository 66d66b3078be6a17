// Static-pivot sparse LU of each independent sub-circuit on gfx950, with
// the Newton update and its norms: the refactor-and-solve that replaces
// N_LAS_AmesosSolver::solve (KLU, N_LAS_AmesosSolver.C:231-470) for every
// Newton iteration after setup.
//
// One workgroup per component.  The component's filled factor pattern and
// its solution vector sit in LDS when they fit (else in a global-memory
// block of their own).  The task lists are level-scheduled: every task of a
// level is independent of the others, so the workgroup runs a level's tasks
// in parallel, one task per thread, and a barrier separates levels.  A task
// is a dot product of earlier values, summed by one thread in ascending
// order, so results do not depend on the launch or on other components.
//
// Static pivots are accepted when the solve is backward stable: every
// pivot nonzero and every factor finite, and the normwise backward error of
// the solution, ||J dx - rhs|| / (||J|| ||dx|| + ||rhs||) (infinity norms,
// the residual taken with the unfactored values), at most 1e-12 -- the
// bound partial pivoting gives in practice (static pivoting with a
// backward-error check, as in Li and Demmel's GESP for SuperLU_DIST).  A
// component that fails is flagged, its iterate left as it was, and the
// dense partial-pivoting kernel launched right after refactors just those.
#include <cfloat>
#include <type_traits>

#include "xg_internal.h"
#include "xg_lu_dev.h"

namespace xg {

namespace {

constexpr int kBlock = 256;
constexpr int kLdsBytes = 144 * 1024;  // factors, vector and task lists
// A component is in LDS when its lists fit at 16 bytes a task and 8 an op
// (sparse_lu_lds_bytes), so none of its numbers exceeds this, and the packed
// lists hold each in 16 bits, a divisor with its sign.
static_assert(kLdsBytes / 8 < 32768, "packed task lists hold 15-bit numbers");

__device__ __forceinline__ double blk_max(double v, double *sv) {
  const int t = threadIdx.x;
  sv[t] = v;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (t < s) sv[t] = fmax(sv[t], sv[t + s]);
    __syncthreads();
  }
  const double r = sv[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ double blk_sum(double v, double *sv) {
  const int t = threadIdx.x;
  sv[t] = v;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (t < s) sv[t] = sv[t] + sv[t + s];
    __syncthreads();
  }
  const double r = sv[0];
  __syncthreads();
  return r;
}

__host__ __device__ constexpr int64_t align16(int64_t b) { return (b + 15) & ~(int64_t)15; }

// A task as the levels run it: destination, divisor, first op and number of
// ops; an op's two operand positions.
struct Task {
  int dst, div, o0, m;
};

// The task lists of one component, level pointers relative to `tasks`.  In
// LDS (kLds) tasks and ops are packed into 8 and 4 bytes (SparseLuArgs::
// ptasks, pops): half the bytes to stage on every solve and one LDS word per
// op.
template <bool kLds>
struct Lists {
  using RawTask = std::conditional_t<kLds, uint2, int4>;
  using RawOp = std::conditional_t<kLds, uint32_t, int2>;
  const RawTask *tasks;
  const RawOp *ops;
  const int32_t *lvp, *lvm, *lvl;  // level -> first task, first mid, first long
  static __device__ __forceinline__ Task task(const RawTask &v) {
    if constexpr (kLds)
      return {(int)(v.x & 0xffff), (int)v.x >> 16, (int)(v.y & 0xffff), (int)(v.y >> 16)};
    else
      return {v.x, v.y, v.z, v.w - v.z};
  }
  // op j of a task, past its end one of its own (whose operands may be read,
  // too), of a task without ops the positions 0
  __device__ __forceinline__ RawOp op_of(const Task &t, int j) const {
    const RawOp v = ops[t.m > 0 ? t.o0 + min(j, t.m - 1) : 0];
    if constexpr (kLds)
      return t.m > 0 ? v : 0;
    else
      return t.m > 0 ? v : RawOp{0, 0};
  }
  static __device__ __forceinline__ int2 op(const RawOp &v) {
    if constexpr (kLds)
      return {(int)(v & 0xffff), (int)(v >> 16)};
    else
      return v;
  }
};

// Finishes a task value: division by the pivot d (factor and backward
// solve; read with the task's operands) and the factor's acceptance checks.
template <int kPhase>
__device__ __forceinline__ void finish_task(const Task &tk, double s, double d, double *val,
                                            double *vec, int &bad) {
  if (kPhase == 0) {
    if (tk.div == kLuFwdTask) {  // a forward-substitution row (y in vec)
      vec[tk.dst] = s;
      return;
    }
    if (tk.div >= 0) {  // (every task of a level or none: skipped as a whole)
      s = divide(s, make_pivot(d));
      bad |= !(fabs(s) <= DBL_MAX);  // infinite or NaN
    } else if (tk.div == -2) {
      bad |= !(fabs(s) > 0.0) || isinf(s);
    }
    val[tk.dst] = s;
  } else {
    vec[tk.dst] = kPhase == 2 ? divide(s, make_pivot(d)) : s;
  }
}

// The levels [L0, L1).  Short tasks (at most four terms): one thread each,
// the terms' operands loaded together, then summed in list order.  Mid
// tasks: eight lanes each, long tasks (rows of supply rails, which touch
// most of the circuit): a wavefront each; lane-strided partial sums folded
// by a fixed tree.  The association is fixed by the plan, so results do
// not depend on the launch.
//
// A level is one dependent step and its length is its latency, so it waits
// for one LDS round trip, the operands': the level bounds are in lanes of
// registers, a thread's first short and first mid task are read two levels
// ahead and their ops one level ahead, kept as read until they are used.
// (Bounds, task, ops and operands in turn were 1700 cycles a level.)  Mid
// tasks start from the last wavefront and long ones from the second, so
// that in a level of few tasks they run beside the short ones.
template <int kPhase, bool kLds>
__device__ __forceinline__ void run_levels(const Lists<kLds> &ls, int L0, int L1, double *val,
                                           double *vec, int &bad) {
  using RawTask = typename Lists<kLds>::RawTask;
  using RawOp = typename Lists<kLds>::RawOp;
  if (L0 >= L1) return;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int mid = (kBlock - 1 - t) >> 3, sub = t & 7;
  const int lng = (wave + kBlock / 64 - 1) % (kBlock / 64);
  const double *src0 = kPhase == 0 ? val : vec;
  // lane i: the bounds of level base + i
  int base = 0, bp = 0, bm = 0, bl = 0;
  auto fill = [&](int L) {
    base = L;
    bp = ls.lvp[min(L + lane, L1)];
    bm = ls.lvm[min(L + lane, L1 - 1)];
    bl = ls.lvl[min(L + lane, L1 - 1)];
  };
  struct Ahead {  // a thread's first short and mid task of a level
    RawTask st, mt;
    bool s_on, m_on;
  };
  auto tasks_of = [&](int L) {
    const int i = min(L, L1 - 1) - base;
    const int k0 = __builtin_amdgcn_readlane(bp, i), km = __builtin_amdgcn_readlane(bm, i),
              kl = __builtin_amdgcn_readlane(bl, i);
    Ahead a;
    a.s_on = k0 + t < km;
    a.m_on = km + mid < kl;
    a.st = ls.tasks[a.s_on ? k0 + t : k0];
    a.mt = ls.tasks[a.m_on ? km + mid : k0];
    return a;
  };
  struct Ops {
    RawOp s[4], m[2];
  };
  auto ops_of = [&](const Ahead &a) {
    const Task st = ls.task(a.st), mt = ls.task(a.mt);
    Ops q;
#pragma unroll
    for (int j = 0; j < 4; ++j) q.s[j] = ls.op_of(st, j);
#pragma unroll
    for (int j = 0; j < 2; ++j) q.m[j] = ls.op_of(mt, sub + 8 * j);
    return q;
  };
  auto short_task = [&](const Task &tk, const RawOp *raw, bool on) {
    const double *src = kPhase == 0 && tk.div == kLuFwdTask ? vec : src0;
    double a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int2 q = ls.op(raw[j]);
      a[j] = val[q.x];
      b[j] = src[q.y];
    }
    double s = src[tk.dst];
    const double d = val[max(tk.div, 0)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double n = s - a[j] * b[j];
      s = j < tk.m ? n : s;
    }
    if (on) finish_task<kPhase>(tk, s, d, val, vec, bad);
  };
  auto mid_task = [&](const Task &tk, const RawOp *raw) {
    const double *src = kPhase == 0 && tk.div == kLuFwdTask ? vec : src0;
    const double d = val[max(tk.div, 0)], s0 = src[tk.dst];
    double p = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool in = sub + 8 * j < tk.m;
      const int2 q = ls.op(raw[j]);
      const double n = p + val[q.x] * src[q.y];
      p = in ? n : p;
    }
    for (int o = sub + 16; o < tk.m; o += 8) {
      const int2 r = ls.op(ls.ops[tk.o0 + o]);
      p = p + val[r.x] * src[r.y];
    }
    p = sum8(p);
    if (sub == 0) finish_task<kPhase>(tk, s0 - p, d, val, vec, bad);
  };
  fill(L0);
  Ahead a0 = tasks_of(L0), a1 = tasks_of(L0 + 1);
  Ops q0 = ops_of(a0);
  for (int L = L0; L < L1; ++L) {
    if (L - base > 60) fill(L);
    const int i = L - base;
    const int k0 = __builtin_amdgcn_readlane(bp, i), km = __builtin_amdgcn_readlane(bm, i),
              kl = __builtin_amdgcn_readlane(bl, i), k1 = __builtin_amdgcn_readlane(bp, i + 1);
    const Ops q1 = ops_of(a1);
    const Ahead a2 = tasks_of(L + 2);
    if (k0 + (t & ~63) < km) short_task(ls.task(a0.st), q0.s, a0.s_on);
    for (int k = k0 + t + kBlock; k < km; k += kBlock) {
      const Task tk = ls.task(ls.tasks[k]);
      RawOp q[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) q[j] = ls.op_of(tk, j);
      short_task(tk, q, true);
    }
    if (a0.m_on) mid_task(ls.task(a0.mt), q0.m);
    for (int k = km + mid + kBlock / 8; k < kl; k += kBlock / 8) {
      const Task tk = ls.task(ls.tasks[k]);
      RawOp q[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) q[j] = ls.op_of(tk, sub + 8 * j);
      mid_task(tk, q);
    }
    for (int k = kl + lng; k < k1; k += kBlock / 64) {
      const Task tk = ls.task(ls.tasks[k]);
      const double *src = kPhase == 0 && tk.div == kLuFwdTask ? vec : src0;
      const double d = val[max(tk.div, 0)], s0 = src[tk.dst];
      double p = 0.0;
#pragma unroll 4
      for (int o = lane; o < tk.m; o += 64) {
        const int2 q = ls.op(ls.ops[tk.o0 + o]);
        p = p + val[q.x] * src[q.y];
      }
      p = wave_sum(p);
      if (lane == 0) finish_task<kPhase>(tk, s0 - p, d, val, vec, bad);
    }
    __syncthreads();
    a0 = a1;
    a1 = a2;
    q0 = q1;
  }
}

// Lays the Jacobian out per component in entry order and the right-hand
// side in position order, so that each component's workgroup reads its
// inputs contiguously.
__global__ void __launch_bounds__(kBlock)
    permute_kernel(int32_t n_ent, int32_t n_nodes, const int32_t *ent_k,
                   const int32_t *prow, const double *J, const double *rhs,
                   double *Jp, double *bp, const int32_t *gate) {
  if (gate && *gate) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n_ent) Jp[i] = J[ent_k[i]];
  if (i < n_nodes) bp[i] = rhs[prow[i]];
}

template <bool kLds>
__global__ void __launch_bounds__(kBlock) sparse_lu_kernel(SparseLuArgs a) {
  __shared__ __align__(16) char lds[kLds ? kLdsBytes : 16];
  __shared__ double sv[kBlock];
  const int c = blockIdx.x;
  const int t = threadIdx.x;
  // (the component in one load, beside the stop word and its activity)
  const LuComp q = a.comp[c];
  const bool off = a.active && !a.active[c];
  if (a.gate && *a.gate) return;
  if (q.in_lds != (kLds ? 1 : 0)) return;  // the other form
  const int beg = q.beg, n = q.n;
  const int64_t nv = q.nv;
  double *stats = a.stats + 4 * (size_t)c;
  if (off) {
    if (t == 0) {
      stats[0] = 0.0;
      stats[1] = 0.0;
      stats[2] = 0.0;
      stats[3] = 0.0;
      a.fallback[c] = 0;
    }
    return;
  }
  if (q.front) {  // the dense-front kernels solve it
    if (t == 0) a.fallback[c] = 0;
    return;
  }
  if (!q.ok) {  // structurally singular under matching: dense kernel
    if (t == 0) a.fallback[c] = 1;
    return;
  }
  const int L0 = q.L0, nlev = q.nlev, tbase = q.tbase, ntask = q.ntask, obase = q.obase,
            nops = q.nops;
  double *val, *vec;
  Lists<kLds> ls{};
  if (kLds) {
    // stage: [values][vector][tasks][ops][level pointers]
    char *p = lds;
    val = (double *)p;
    p += align16(nv * 8);
    vec = (double *)p;
    p += align16((int64_t)n * 8);
    uint2 *tk = (uint2 *)p;
    p += align16((int64_t)ntask * 8);
    uint32_t *op = (uint32_t *)p;
    p += align16((int64_t)nops * 4);
    int32_t *lvp = (int32_t *)p;
    int32_t *lvm = lvp + nlev + 1;
    int32_t *lvl = lvm + nlev;
#pragma unroll 8
    for (int k = t; k < ntask; k += kBlock) tk[k] = a.ptasks[tbase + k];
#pragma unroll 8
    for (int k = t; k < nops; k += kBlock) op[k] = a.pops[obase + k];
    for (int k = t; k <= nlev; k += kBlock) lvp[k] = a.lv_ptr[L0 + k] - tbase;
    for (int k = t; k < nlev; k += kBlock) {
      lvm[k] = a.lv_mid[L0 + k] - tbase;
      lvl[k] = a.lv_long[L0 + k] - tbase;
    }
    ls.tasks = (const typename Lists<kLds>::RawTask *)tk;
    ls.ops = (const typename Lists<kLds>::RawOp *)op;
    ls.lvp = lvp;
    ls.lvm = lvm;
    ls.lvl = lvl;
  } else {
    val = a.val_work + q.voff;
    vec = a.vec_work + beg;
    // global lists: level pointers and ops stay absolute
    ls.tasks = (const typename Lists<kLds>::RawTask *)a.tasks;
    ls.ops = (const typename Lists<kLds>::RawOp *)a.ops;
    ls.lvp = a.lv_ptr + L0;
    ls.lvm = a.lv_mid + L0;
    ls.lvl = a.lv_long + L0;
  }
  const int32_t *qcol = a.qcol + beg;
  // the component's Jacobian entries and right-hand side, already laid out
  // contiguously by the permute kernel
  const int eb = q.eb, ne = q.ne;
  const double *jp = a.Jp + eb, *bp = a.bp + beg;
  const int32_t *epos = a.ent_pos + eb, *ecol = a.ent_col + eb, *ers = a.ent_rs + beg + c;
  for (int64_t e = t; e < nv; e += kBlock) val[e] = 0.0;
  __syncthreads();
#pragma unroll 8
  for (int j = t; j < ne; j += kBlock) val[epos[j]] = jp[j];
  double rmax = 0.0;
  for (int i = t; i < n; i += kBlock) {
    const double r = bp[i];
    vec[i] = r;
    rmax = fmax(rmax, fabs(r));
  }
  const double max_rhs = blk_max(rmax, sv);  // includes the barriers
  // ---- factor
  const int f1 = q.f1, s1 = q.s1;
  int bad = 0;
  run_levels<0>(ls, 0, f1, val, vec, bad);
  if (__syncthreads_or(bad)) {
    if (t == 0) a.fallback[c] = 1;
    return;
  }
  // ---- L y = P b (unit diagonal), then U x' = y, in place
  run_levels<1>(ls, f1, s1, val, vec, bad);
  run_levels<2>(ls, s1, nlev, val, vec, bad);
  // ---- backward error of the solution against the unfactored rows
  // (rows of more than kWaveRow entries, the supply rails, by a wavefront
  // each: in one thread a 600-entry row took 13 us of the 70)
  constexpr int kWaveRow = 32;
  double rm = 0.0, am = 0.0, xm = 0.0;
  for (int i0 = 0; i0 < n; i0 += kBlock) {
    const int i = i0 + t;
    const int j0 = i < n ? ers[i] : 0, j1 = i < n ? ers[i + 1] : 0;
    const bool wide = j1 - j0 > kWaveRow;
    if (i < n) xm = fmax(xm, fabs(vec[i]));
    if (i < n && !wide) {
      double r = bp[i], as = 0.0;
#pragma unroll 8
      for (int j = j0; j < j1; ++j) {
        const double v = jp[j];
        r = r - v * vec[ecol[j]];
        as = as + fabs(v);
      }
      rm = fmax(rm, fabs(r));
      am = fmax(am, as);
    }
    unsigned long long mask = __ballot(wide);
    while (mask) {  // this wavefront's wide rows
      const int l = __ffsll(mask) - 1;
      mask &= mask - 1;
      const int w0 = __builtin_amdgcn_readlane(j0, l), w1 = __builtin_amdgcn_readlane(j1, l);
      double r = 0.0, as = 0.0;
#pragma unroll 4
      for (int j = w0 + (t & 63); j < w1; j += 64) {
        const double v = jp[j];
        r = r + v * vec[ecol[j]];
        as = as + fabs(v);
      }
      r = wave_sum(r);
      as = wave_sum(as);
      rm = fmax(rm, fabs(bp[__builtin_amdgcn_readlane(i, l)] - r));
      am = fmax(am, as);
    }
  }
  rm = blk_max(rm, sv);
  am = blk_max(am, sv);
  xm = blk_max(xm, sv);
  if (!(rm <= a.max_berr * (am * xm + max_rhs))) {  // also NaN / infinite
    if (t == 0) a.fallback[c] = 1;
    return;
  }
  // ---- Newton update x += dx and the weighted RMS norm of dx
  // (N_NLS_DampedNewton.C:311-335)
  double acc = 0.0;
  for (int i = t; i < n; i += kBlock) {
    const int g = qcol[i];
    const double dx = vec[i];
    const double w = a.reltol * fmax(fabs(a.wa[g]), fabs(a.wb[g])) + a.abstol;
    const double q = dx / w;
    acc = acc + q * q;
    a.x[g] = a.x[g] + dx;
  }
  const double ss = blk_sum(acc, sv);
  if (t == 0) {
    stats[0] = max_rhs;
    stats[1] = sqrt(ss / n);
    stats[2] = 0.0;
    stats[3] = (double)n;
    a.fallback[c] = 0;
  }
}

}  // namespace

// The lists count at their unpacked size: twice what the kernel lays out, so
// that the packed numbers fit (above).  Components between the two counts
// take the fronts or the lists in global memory; whether the packed lists in
// LDS would be faster there has not been measured.
int64_t sparse_lu_lds_bytes(int64_t n, int64_t fnnz, int64_t tasks, int64_t ops,
                            int64_t levels) {
  return align16(fnnz * 8) + align16(n * 8) + tasks * 16 + align16(ops * 8) +
         (3 * levels + 1) * 4;
}

int64_t sparse_lu_lds_budget() { return kLdsBytes; }

hipError_t launch_sparse_lu(const SparseLuArgs &a, hipStream_t s) {
  if (a.n_comp == 0) return hipSuccess;
  const int64_t nperm = a.n_ent > a.n_nodes ? a.n_ent : a.n_nodes;
  if (nperm > 0)
    hipLaunchKernelGGL(permute_kernel, dim3((unsigned)((nperm + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, s, a.n_ent, a.n_nodes, a.ent_k, a.prow, a.J,
                       a.rhs, a.Jp, a.bp, a.gate);
  hipLaunchKernelGGL(sparse_lu_kernel<true>, dim3(a.n_comp), dim3(kBlock), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !a.any_global) return e;
  hipLaunchKernelGGL(sparse_lu_kernel<false>, dim3(a.n_comp), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

}  // namespace xg
