// quot.h -- quotients, square roots and t^1.5 of the flux kernels.
#pragma once
#include "cosahip_internal.h"

namespace cosahip {

// ------------------------------------------------------------------------
// Quotients and square roots of the face arithmetic.  The fluxes are bound by
// FP64 instruction issue, and a third of their instructions were divisions
// and square roots: eleven for each division (two that scale for extreme
// exponents and one that fixes specials up), about twenty for a root.  Here, in FP64:
//   * a divisor is inverted once, by Newton-Raphson to the last bits, and
//     every quotient by it takes three instructions: q = n y, then Markstein's
//     correction q + (n - q d) y, which rounds to the correctly rounded n / d
//     (IBM J. Res. Dev. 34 (1990) 111-119); the correction is written as
//     -(q d - n) y + q, which keeps the sign of an exact zero n (d > 0);
//   * sqrt(x) comes from the hardware's 1 / sqrt(x) by Goldschmidt's iteration
//     and two of the same corrections; the refined 1 / sqrt(x) squared is the
//     start of the inverse of x itself, which saves that its own.
// The bits are those of the division and the root for operands without
// extreme exponents (states and their differences: no subnormals, no
// overflow; below 1e-290 a quotient keeps its absolute, not its relative
// rounding).  Where the flow state has failed already they give NaN: for a zero
// or negative divisor, for which the division gives an infinity, and for an
// infinite operand, for which division, root and power give an infinity or zero.
// FP32 and the contracted build use the operators.
// Residual of 48 uneven blocks (with the end tests of muscl_face below):
// VALU instructions 439 M -> 334 M, level 1 1230 -> 1128 us, level 2 160 -> 133;
// HB O-grid 180 -> 155 us.  It is now bound by the latency of each plane's
// loads behind its barriers at three waves per SIMD (162 VGPRs): without any
// Roe flux or limiter division it still took 931 us.  Loading the next plane
// or the metrics ahead cost the third wave and lost (1180-1450 us).
#ifdef COSAHIP_CONTRACTED
constexpr bool FACE_QUOT = false;
#else
constexpr bool FACE_QUOT = true;
#endif
template <typename T>
struct Divisor {
  T d, y;
  __device__ __forceinline__ Divisor() {}
  __device__ __forceinline__ explicit Divisor(T d_) : d(d_), y(0) {
    if constexpr (FACE_QUOT && sizeof(T) == 8) {
      y = __builtin_amdgcn_rcp(d);
      y = fma(fma(-d, y, 1.0), y, y);
      y = fma(fma(-d, y, 1.0), y, y);
    }
  }
  // y0: an approximate inverse of d with at least half its bits right
  __device__ __forceinline__ Divisor(T d_, T y0) : d(d_), y(y0) {
    if constexpr (FACE_QUOT && sizeof(T) == 8) y = fma(fma(-d, y, 1.0), y, y);
  }
  // y: the correctly rounded inverse (a run constant's, from the host)
  static __device__ __forceinline__ Divisor constant(T d_, double y_) {
    Divisor r;
    r.d = d_;
    r.y = (T)y_;
    return r;
  }
  __device__ __forceinline__ T of(T n) const {
    if constexpr (FACE_QUOT && sizeof(T) == 8) {
      const T q = n * y;
      return fma(-fma(q, d, -n), y, q);
    } else {
      return n / d;
    }
  }
};
// sqrt(x); rs: about 1 / sqrt(x) (FP64)
template <typename T>
__device__ __forceinline__ T face_sqrt(T x, T& rs) {
  if constexpr (FACE_QUOT && sizeof(T) == 8) {
    const T y = __builtin_amdgcn_rsq(x);
    T g = x * y, h = y * 0.5;
    const T r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    rs = h + h;
    return g;
  } else {
    rs = 0;
    return sqrt(x);
  }
}

// t^1.5 as t sqrt(t) with the rounding errors of both steps added back: s =
// sqrt(t) is short by (t - s^2) / 2s, p = t s by t s - p, each exact or nearly
// so from a fused multiply-add, so the sum is within 0.51 ulp of t^1.5 -- the
// library's pow is within one -- in a dozen instructions instead of some two
// hundred.  0 gives 0, a negative t NaN, as pow does.
// k-omega wing, level 1 (2.1 M cells): the spectral radii, seven of these a
// cell, 224 -> 149 us (105 since the smoothing's powers are out of their
// kernel); the viscous faces, with the quotients of viscous_face, 209/204/192
// -> 202/196/184 us -- they are bound by their loads.
template <typename T>
__device__ __forceinline__ T pow32(T t) {
  const T s = sqrt(t);
  const T ds = s > T(0) ? fma(-s, s, t) / (s + s) : T(0), p = t * s;
  return p + fma(t, ds, fma(t, s, -p));
}
__device__ __forceinline__ double pow32(double t) {
  double rs;
  const double s = face_sqrt(t, rs), p = t * s;
  const double e = fma(t, fma(-s, s, t) * (rs * 0.5), fma(t, s, -p));
  return t == 0.0 ? 0.0 : p + e;
}

}  // namespace cosahip
