// sincos.hpp -- sine and cosine in f64 for the Helmholtz pair kernel.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace fmmh {
namespace dev {

// x = n pi/2 + t + tl, |t| <= pi/4, with pi/2 as the sum of two doubles (Cody and Waite), tl what
// rounding t left out; sine and cosine of t by polynomials in t^2 through the Chebyshev points
// of [0, (pi/4)^2] (errors 1.2e-20 and 1.3e-18), the last two terms of each summed with the
// rounding of the first carried along; the quadrant selects and signs.  For |x| < 2^31, far
// beyond any k r of a leaf pair.  Against long double over (0, 6), (0, 60) and (0, 600): at most
// 0.77 ulp, rms 0.293 (the math library's: 0.78 and 0.294; without tl and the carried rounding
// 1.54 and 0.418).

// The sine and cosine of the reduced argument, and its quadrant n (its low two bits).
__host__ __device__ __forceinline__ uint32_t sincos_reduced(double x, double *s, double *c) {
  constexpr double kShift = 6755399441055744.0;  // 1.5 2^52: the sum's low bits are rint(x 2/pi)
  const double m = std::fma(x, 0.6366197723675814, kShift), n = m - kShift;
  const uint32_t q = uint32_t(__builtin_bit_cast(uint64_t, m));
  const double t1 = std::fma(-n, 1.5707963267948966, x);  // exact
  const double t = std::fma(-n, 6.123233995736766e-17, t1), tl = std::fma(-n, 6.123233995736766e-17, t1 - t);
  const double z = t * t;
  double ps = std::fma(z, -7.586697117706918e-13, 1.6058531618986147e-10);
  ps = std::fma(z, ps, -2.5052106232447578e-08);
  ps = std::fma(z, ps, 2.7557319219339167e-06);
  ps = std::fma(z, ps, -0.00019841269841265065);
  ps = std::fma(z, ps, 0.008333333333333331);
  ps = std::fma(z, ps, -0.16666666666666666);
  double pc = std::fma(z, -1.1382632425521717e-11, 2.08761462684032e-09);
  pc = std::fma(z, pc, -2.7557317271729793e-07);
  pc = std::fma(z, pc, 2.480158729876569e-05);
  pc = std::fma(z, pc, -0.0013888888888887398);
  pc = std::fma(z, pc, 0.041666666666666664);
  // 1 - z / 2, and what its rounding left out
  const double w = std::fma(-0.5, z, 1.0), e = std::fma(-0.5, z, 1.0 - w);
  *s = t + std::fma(t * z, ps, w * tl);
  *c = w + std::fma(z * z, pc, std::fma(-t, tl, e));
  return q;
}

__host__ __device__ __forceinline__ void sincos_f64(double x, double *s, double *c) {
  double st, ct;
  const uint32_t q = sincos_reduced(x, &st, &ct);
  const double sv = (q & 1) ? ct : st, cv = (q & 1) ? st : ct;
  *s = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, sv) ^ (uint64_t(q & 2) << 62));
  *c = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, cv) ^ (uint64_t((q + 1) & 2) << 62));
}

}  // namespace dev
}  // namespace fmmh
