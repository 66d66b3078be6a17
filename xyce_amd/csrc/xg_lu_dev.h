// Device arithmetic shared by the LU kernels (xg_lu.hip, xg_front.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace xg {

// p[i], or 0 where it may not be read (p[0] may): a select, no branch, so
// that a run of these loads is in flight together (behind `cond ? p[i] : 0`
// with a short-circuit the compiler waits for each one).
__device__ __forceinline__ double load_if(bool ok, const double *p, int64_t i) {
  const double v = p[ok ? i : 0];
  return ok ? v : 0.0;
}

// Division by a pivot shared by many rows: the pivot's mantissa p, its
// reciprocal r and minus its exponent, then per row a quotient and one
// correction with the exact remainder (four operations instead of the ~11 of
// a full division; the last bit's error is that of one rounding but for
// rare double roundings).  Scaling by the exponent keeps the whole range.
// Every form below divides this way, so all give the same bits.
struct Pivot {
  double p, r;
  int e;
};
__device__ __forceinline__ Pivot make_pivot(double v) {
  const double p = __builtin_amdgcn_frexp_mant(v);
  return {p, 1.0 / p, -__builtin_amdgcn_frexp_exp(v)};
}
__device__ __forceinline__ double divide(double a, const Pivot &v) {
  const double x = __builtin_amdgcn_ldexp(a, v.e);
  const double q = x * v.r;
  return fma(fma(-q, v.p, x), v.r, q);
}

__device__ __forceinline__ double read_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// Sums over 8 lanes and over the wavefront, the same bits in every lane:
// neighbours, then pairs, quads and halves (each step adds two mirror
// images), then the four rows of 16.
template <int kCtrl>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return v + __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, kCtrl, 0xf, 0xf, false),
                              __builtin_amdgcn_update_dpp(lo, lo, kCtrl, 0xf, 0xf, false));
}
__device__ __forceinline__ double sum8(double v) {
  return dpp_add<0x141>(dpp_add<0x4e>(dpp_add<0xb1>(v)));
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x140>(sum8(v));
  return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

}  // namespace xg
