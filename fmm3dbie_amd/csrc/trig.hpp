// sin and cos of FP64 arguments of bounded size, for the Helmholtz kernel evaluations
// (sincos_turns: far sums; sincos_pi: quadrature, whose kernels take its two steps one by one in
// sincos_near, common.hpp) and for callers of the library on the host (sincos_red, which no
// kernel uses).
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

// Largest |x| for each: n = rint(2x/pi) stays below 2^20, where the three-part reductions
// below are accurate to rounding.  The host checks |k| times the largest
// distance of a computation against it.
constexpr double SINCOS_RED_MAX = 1.6e6;

// sin x and cos x for |x| <= SINCOS_RED_MAX.
// x = n pi/2 + y with n = rint(2x/pi): y from three fused multiply-adds with pi/2 split
// into three doubles p1 + p2 + p3 (Cody and Waite's additive reduction; the split is
// computed from the decimal digits of pi and equals pi/2 to 5.6e-50).  sin y and cos y
// come from their Taylor series through y^15 and y^16 (coefficients +-1/k!, rounded to
// nearest): on |y| <= pi/4 the first omitted terms are below 5e-17 and 3e-18.  The
// quadrant n mod 4 then maps (sin y, cos y) to (sin x, cos x).
__host__ __device__ __forceinline__ void sincos_red(double x, double& s, double& c) {
  const double n = rint(x * 0x1.45f306dc9c883p-1);  // 2/pi
  double y = fma(-n, 0x1.921fb54442d18p+0, x);        // p1
  y = fma(-n, 0x1.1a62633145c07p-54, y);              // p2
  y = fma(-n, -0x1.f1976b7ed8fbcp-110, y);            // p3
  const double z = y * y;
  double ps = -0x1.ae7f3e733b81fp-41;  // -1/15!
  ps = fma(ps, z, 0x1.6124613a86d09p-33);   // 1/13!
  ps = fma(ps, z, -0x1.ae64567f544e4p-26);  // -1/11!
  ps = fma(ps, z, 0x1.71de3a556c734p-19);   // 1/9!
  ps = fma(ps, z, -0x1.a01a01a01a01ap-13);  // -1/7!
  ps = fma(ps, z, 0x1.1111111111111p-7);    // 1/5!
  ps = fma(ps, z, -0x1.5555555555555p-3);   // -1/3!
  const double sn = fma(ps * z, y, y);
  double pc = 0x1.ae7f3e733b81fp-45;        // 1/16!
  pc = fma(pc, z, -0x1.93974a8c07c9dp-37);  // -1/14!
  pc = fma(pc, z, 0x1.1eed8eff8d898p-29);   // 1/12!
  pc = fma(pc, z, -0x1.27e4fb7789f5cp-22);  // -1/10!
  pc = fma(pc, z, 0x1.a01a01a01a01ap-16);   // 1/8!
  pc = fma(pc, z, -0x1.6c16c16c16c17p-10);  // -1/6!
  pc = fma(pc, z, 0x1.5555555555555p-5);    // 1/4!
  pc = fma(pc, z, -0.5);                    // -1/2!
  const double cn = fma(pc, z, 1.0);
  const int q = (int)n & 3;  // n mod 4, also for negative n
  const double sq = (q & 1) ? cn : sn, cq = (q & 1) ? sn : cn;
  s = (q & 2) ? -sq : sq;
  c = ((q + 1) & 2) ? -cq : cq;
}

// k / pi as a sum of two doubles (host): r * (hi + lo) is k r in half turns
inline void half_turns(double k, double& hi, double& lo) {
  constexpr double ih = 0x1.45f306dc9c883p-2, il = -0x1.6b01ec5417056p-56;  // 1 / pi
  hi = k * ih;
  lo = std::fma(k, ih, -hi) + k * il;
}

// sin(k r) and cos(k r) for the far sums, r (khi + klo) = k r / pi (half_turns), k r <=
// SINCOS_RED_MAX; both values have to be multiplied by -1 where neg is set (a caller with a
// further factor puts the sign there).
// The argument is reduced to the nearest multiple of pi: adding 1.5 * 2^52 rounds it to a
// whole number n of half turns, whose parity is the last bit of the sum, and y = r (khi +
// klo) - n (|y| <= 1/2) takes two fused multiply-adds with no rounding of k r itself.
// sin(pi y) / y and cos(pi y) are polynomials of degree 8 in y^2, minimax on [0, 1/4] (Remez
// exchange in 300 bits; errors 1.6e-19 and 3.9e-18).  A reduction by pi needs neither the
// swap of sine and cosine nor the quadrant signs of one by pi/2 at the same polynomial work.
// Error against 60-digit arithmetic over k r up to SINCOS_RED_MAX: at most 3.9e-16; over k r up to 40 in
// root mean square 0.9e-16, where sincos_red of the rounded product k * r has 6.5e-16 (the product's
// rounding).
__host__ __device__ __forceinline__ void sincos_turns(double r, double khi, double klo, double& s, double& c,
                                                      bool& neg) {
  const double m = fma(r, khi, 0x1.8p52);
  const double n = m - 0x1.8p52;
  const double y = fma(r, klo, fma(r, khi, -n));
  const double z = y * y;
  double ps = 0x1.9c88754152556p-21;
  ps = fma(ps, z, -0x1.6f7481d5954e2p-16);
  ps = fma(ps, z, 0x1.e8f33b4e47ba7p-12);
  ps = fma(ps, z, -0x1.e3074d575a249p-8);
  ps = fma(ps, z, 0x1.50783483f78e5p-4);
  ps = fma(ps, z, -0x1.32d2cce6248a9p-1);
  ps = fma(ps, z, 0x1.466bc6775a9f9p+1);
  ps = fma(ps, z, -0x1.4abbce625be51p+2);
  ps = fma(ps, z, 0x1.921fb54442d18p+1);
  s = ps * y;
  double pc = 0x1.1679716d61ddbp-18;
  pc = fma(pc, z, -0x1.b69582daed135p-14);
  pc = fma(pc, z, 0x1.f9d254890ff5fp-10);
  pc = fma(pc, z, -0x1.a6d1efc969016p-6);
  pc = fma(pc, z, 0x1.e1f506813c9e7p-3);
  pc = fma(pc, z, -0x1.55d3c7e3bfc44p+0);
  pc = fma(pc, z, 0x1.03c1f081b5993p+2);
  pc = fma(pc, z, -0x1.3bd3cc9be45dbp+2);
  c = fma(pc, z, 1.0);
  union {
    double d;
    uint64_t u;
  } b;
  b.d = m;
  neg = b.u & 1;
}

// sin x and cos x for |x| <= pi/2 without a reduction: minimax polynomials (sin x / x - 1) / x^2
// and (cos x - 1) / x^2 of degree 7 in x^2 (Remez exchange in 300 bits, errors 2.0e-19 and
// 4.3e-18).
// The coefficients are kept in scalar registers (scalar_const): as literals each costs two
// vector moves at every use, as many instructions as the polynomials themselves.
__host__ __device__ __forceinline__ double scalar_const(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(x));
#endif
  return x;
}
__host__ __device__ __forceinline__ void sincos_half_pi(double x, double& s, double& c) {
  const double z = x * x;
  double ps = scalar_const(0x1.87cf34cb45316p-49);
  ps = fma(ps, z, scalar_const(-0x1.ae3f72f9ed52ap-41));
  ps = fma(ps, z, scalar_const(0x1.6123bb933d336p-33));
  ps = fma(ps, z, scalar_const(-0x1.ae645485a9287p-26));
  ps = fma(ps, z, scalar_const(0x1.71de3a51d914ep-19));
  ps = fma(ps, z, scalar_const(-0x1.a01a01a012a97p-13));
  ps = fma(ps, z, scalar_const(0x1.1111111111098p-7));
  ps = fma(ps, z, scalar_const(-0x1.5555555555555p-3));
  s = fma(ps, z * x, x);
  double pc = scalar_const(0x1.9f4e7cd1ca798p-45);
  pc = fma(pc, z, scalar_const(-0x1.93525f737d4a0p-37));
  pc = fma(pc, z, scalar_const(0x1.1eece69a30ce8p-29));
  pc = fma(pc, z, scalar_const(-0x1.27e4f99a6d27fp-22));
  pc = fma(pc, z, scalar_const(0x1.a01a0199f59b7p-16));
  pc = fma(pc, z, scalar_const(-0x1.6c16c16c0b99ap-10));
  pc = fma(pc, z, scalar_const(0x1.555555555541ep-5));
  pc = fma(pc, z, scalar_const(-0x1.ffffffffffffdp-2));
  c = fma(pc, z, 1.0);
}

// x = n pi + y, |y| <= pi/2 (the rounding of x / pi aside), |x| <= SINCOS_RED_MAX: returns n.  Three-part
// reduction as in sincos_red.
__host__ __device__ __forceinline__ double pi_reduce(double x, double& y) {
  const double n = rint(x * 0x1.45f306dc9c883p-2);  // 1/pi
  y = fma(-n, 0x1.921fb54442d18p+1, x);
  y = fma(-n, 0x1.1a62633145c07p-53, y);
  y = fma(-n, -0x1.f1976b7ed8fbcp-109, y);
  return n;
}

// sin x and cos x for |x| <= SINCOS_RED_MAX: pi_reduce, sincos_half_pi and the sign of n's parity.
__host__ __device__ __forceinline__ void sincos_pi(double x, double& s, double& c) {
  double y;
  const bool odd = (int)pi_reduce(x, y) & 1;
  sincos_half_pi(y, s, c);
  s = odd ? -s : s;
  c = odd ? -c : c;
}
