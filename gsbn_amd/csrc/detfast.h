/*
 * detfast.h -- the float results of detmath.h and philox.h from shorter
 * double sequences, bit for bit, for the kernels that draw, exponentiate and
 * take logarithms per unit and are bound by the issue of these operations.
 *
 * The float results of gsbn_expf, gsbn_logf and gsbn_draw_unit are roundings
 * of a double value to 24 bits.  Here the value is first computed by a
 * shorter sequence (fused multiply-adds, a hardware reciprocal or reciprocal
 * square root with one Newton step, fewer series terms) whose relative
 * distance from the full sequence is below 2e-14.  A double whose 29 bits
 * below the float's last bit are at least GSBN_GUARD units away from the
 * midpoint between two floats rounds to the same float as every value within
 * GSBN_GUARD units (2.3e-13 to 4.5e-13 relative, more than ten times that
 * distance), so its rounding is the rounding of the full sequence's value;
 * the others, about one in 10^5, run the full sequence.  (Compared on gfx950
 * for every float argument of exp and log and for 2^32 pairs of 24-bit words
 * of the normal deviate: no bit differs; the deviate's largest distance is
 * 5.3e-15.)  Measured: the recall's population step, 8192 cues of 100 x 100
 * units, 1100 us -> 857 us.
 */
#ifndef GSBN_DETFAST_H
#define GSBN_DETFAST_H

#include <stdint.h>

#include "detmath.h"
#include "philox.h"

/* The full sequences of detmath.h for the fallbacks: the series are loops
 * over a table, so that their constants stay out of the kernels' registers
 * (inlined and unrolled, they made the batched population kernel spill 74). */
template <int N>
GSBN_HD GSBN_INLINE double gsbn_horner(const double (&c)[N], double x) {
  double p = c[0];
#if defined(__HIP_DEVICE_COMPILE__)
#pragma clang loop unroll(disable)
#endif
  for (int i = 1; i < N; ++i) p = p * x + c[i];
  return p;
}

/* gsbn_exp */
GSBN_HD GSBN_INLINE double gsbn_exp_cold(double x) {
  if (x != x) return x;
  if (x > 709.78) return gsbn_bitsd(0x7ff0000000000000ULL);
  if (x < -745.2) return 0.0;
  const double kd = gsbn_rint_small(x * 1.44269504088896338700e+00);
  const int k = (int)kd;
  const double r = (x - kd * 6.93147180369123816490e-01) - kd * 1.90821492927058770002e-10;
  static const double c[14] = {1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0,
                               1.0 / 3628800.0,    1.0 / 362880.0,    1.0 / 40320.0,
                               1.0 / 5040.0,       1.0 / 720.0,       1.0 / 120.0,
                               1.0 / 24.0,         1.0 / 6.0,         0.5,
                               1.0,                1.0}; /* 1/13! .. 1/0! */
  const double p = gsbn_horner(c, r);
  const int k1 = k / 2, k2 = k - k1;
  return (p * gsbn_bitsd((uint64_t)(int64_t)(k1 + 1023) << 52)) *
         gsbn_bitsd((uint64_t)(int64_t)(k2 + 1023) << 52);
}

/* gsbn_log of a float argument (never subnormal as a double) */
GSBN_HD GSBN_INLINE double gsbn_log_cold(double x) {
  if (x != x) return x;
  if (x < 0.0) return gsbn_bitsd(0x7ff8000000000000ULL);
  if (x == 0.0) return gsbn_bitsd(0xfff0000000000000ULL);
  const uint64_t b = gsbn_dbits(x);
  if ((b >> 52) == 0x7ff) return x; /* +inf */
  int e = (int)(b >> 52) - 1023;
  double m = gsbn_bitsd((b & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL);
  if (m > 1.41421356237309504880) {
    m = m * 0.5;
    e += 1;
  }
  const double f = m - 1.0;
  const double s = f / (2.0 + f);
  const double z = s * s;
  static const double c[12] = {1.0 / 23.0, 1.0 / 21.0, 1.0 / 19.0, 1.0 / 17.0,
                               1.0 / 15.0, 1.0 / 13.0, 1.0 / 11.0, 1.0 / 9.0,
                               1.0 / 7.0,  1.0 / 5.0,  1.0 / 3.0,  1.0};
  const double logm = 2.0 * s * gsbn_horner(c, z);
  const double ed = (double)e;
  return ed * 6.93147180369123816490e-01 + (ed * 1.90821492927058770002e-10 + logm);
}

/* gsbn_cos2pi */
GSBN_HD GSBN_INLINE double gsbn_cos2pi_cold(double u) {
  const double v = u - gsbn_rint_small(u);
  double a = v < 0.0 ? -v : v;
  double sign = 1.0;
  if (a > 0.25) {
    a = 0.5 - a;
    sign = -1.0;
  }
  const double two_pi = 6.28318530717958647692;
  double r;
  if (a > 0.125) {
    const double t = two_pi * (0.25 - a), t2 = t * t;
    static const double c[8] = {-1.0 / 355687428096000.0, 1.0 / 1307674368000.0,
                                -1.0 / 6227020800.0,      1.0 / 39916800.0,
                                -1.0 / 362880.0,          1.0 / 5040.0,
                                -1.0 / 120.0,             1.0 / 6.0}; /* -1/17! .. 1/3! */
    r = t - t * t2 * gsbn_horner(c, t2);
  } else {
    const double t = two_pi * a, t2 = t * t;
    static const double c[9] = {1.0 / 6402373705728000.0, -1.0 / 20922789888000.0,
                                1.0 / 87178291200.0,      -1.0 / 479001600.0,
                                1.0 / 3628800.0,          -1.0 / 40320.0,
                                1.0 / 720.0,              -1.0 / 24.0,
                                0.5}; /* 1/18! .. 1/2! */
    r = 1.0 - t2 * gsbn_horner(c, t2);
  }
  return sign * r;
}

/* gsbn_draw_unit's normal of two 24-bit words */
GSBN_HD GSBN_INLINE float gsbn_normal24_cold(uint32_t k1, uint32_t k2) {
  const double inv24 = 5.9604644775390625e-08;
  const double r = gsbn_sqrt(-2.0 * gsbn_log_cold((double)(k1 + 1u) * inv24));
  return (float)(r * gsbn_cos2pi_cold((double)k2 * inv24));
}

#define GSBN_GUARD 2048

GSBN_HD GSBN_INLINE int gsbn_round_safe(double y) {
  const int d = (int)((uint32_t)gsbn_dbits(y) & 0x1fffffffu) - 0x10000000;
  return d > GSBN_GUARD || d < -GSBN_GUARD;
}

/* Seeds of 1/x and 1/sqrt(x), within 2^-24 relative (the instructions are
 * specified to 2^29 units in the last place).  One Newton step on a seed that
 * is off by e leaves e^2 = 3.6e-15 of the reciprocal and 1.5 e^2 = 5.3e-15 of
 * the square root.  A host build can set the seeds' error (GSBN_SEED_ERROR). */
GSBN_HD GSBN_INLINE double gsbn_rcp_seed(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcp(x);
#elif defined(GSBN_SEED_ERROR)
  return (1.0 + GSBN_SEED_ERROR) / x;
#else
  return (double)(1.0f / (float)x);
#endif
}
GSBN_HD GSBN_INLINE double gsbn_rsq_seed(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsq(x);
#elif defined(GSBN_SEED_ERROR)
  return (1.0 + GSBN_SEED_ERROR) / __builtin_sqrt(x);
#else
  return (double)(1.0f / __builtin_sqrtf((float)x));
#endif
}

/* p x + c for a series constant c.  Written out on the device so that c stays
 * in scalar registers: the compiler's two-operand form first copies each
 * constant into the accumulator with two more vector instructions. */
GSBN_HD GSBN_INLINE double gsbn_fmac(double p, double x, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(p), "v"(x), "s"(c));
  return d;
#else
  return __builtin_fma(p, x, c);
#endif
}

/* e^x in double, -87 <= x <= 88: series to r^11 (truncation below 7e-15) */
GSBN_HD GSBN_INLINE double gsbn_exp_short(double x) {
  const double kd = __builtin_rint(x * 1.44269504088896338700e+00);
  double r = __builtin_fma(kd, -6.93147180369123816490e-01, x);
  r = __builtin_fma(kd, -1.90821492927058770002e-10, r);
  double p = 1.0 / 39916800.0;
  p = gsbn_fmac(p, r, 1.0 / 3628800.0);
  p = gsbn_fmac(p, r, 1.0 / 362880.0);
  p = gsbn_fmac(p, r, 1.0 / 40320.0);
  p = gsbn_fmac(p, r, 1.0 / 5040.0);
  p = gsbn_fmac(p, r, 1.0 / 720.0);
  p = gsbn_fmac(p, r, 1.0 / 120.0);
  p = gsbn_fmac(p, r, 1.0 / 24.0);
  p = gsbn_fmac(p, r, 1.0 / 6.0);
  p = gsbn_fmac(p, r, 0.5);
  p = gsbn_fmac(p, r, 1.0);
  p = gsbn_fmac(p, r, 1.0);
  /* p in [0.7, 1.42] and |k| <= 127: the exponent field takes k directly */
  return gsbn_bitsd(gsbn_dbits(p) + ((uint64_t)(uint32_t)(int)kd << 52));
}

/* log x in double for a normal positive float: the same reduction and
 * series, to s^17 (truncation below 1e-15), 1/(m+1) from the seed and one
 * Newton step (4e-15; up to 8e-15 of a logarithm that cancels) */
GSBN_HD GSBN_INLINE double gsbn_log_short(float x) {
  const uint32_t b = gsbn_fbits(x);
  const uint32_t mb = b & 0x7fffffu;
  const int up = mb > 0x3504f3u; /* m above sqrt(2): halve it */
  const double ed = (double)((int)(b >> 23) - 127 + up);
  const double m = (double)gsbn_bitsf(mb | (up ? 0x3f000000u : 0x3f800000u));
  const double den = m + 1.0;
  double y = gsbn_rcp_seed(den);
  y = __builtin_fma(y, __builtin_fma(-den, y, 1.0), y);
  const double s = (m - 1.0) * y;
  const double z = s * s;
  double q = 1.0 / 17.0;
  q = gsbn_fmac(q, z, 1.0 / 15.0);
  q = gsbn_fmac(q, z, 1.0 / 13.0);
  q = gsbn_fmac(q, z, 1.0 / 11.0);
  q = gsbn_fmac(q, z, 1.0 / 9.0);
  q = gsbn_fmac(q, z, 1.0 / 7.0);
  q = gsbn_fmac(q, z, 1.0 / 5.0);
  q = gsbn_fmac(q, z, 1.0 / 3.0);
  const double s2 = s + s;
  return __builtin_fma(ed, 6.93147180559945309417e-01, __builtin_fma(s2 * z, q, s2));
}

/* sin(2 pi i / 2^24) in double for |i| <= 2^22: Taylor series to t^19
 * (truncation below 2e-16 on |t| <= pi/2) */
GSBN_HD GSBN_INLINE double gsbn_sin2pi24(int i) {
  const double t = (double)i * 3.7450702829239286e-07; /* 2 pi / 2^24 */
  const double t2 = t * t;
  double p = -1.0 / 121645100408832000.0;             /* -1/19! */
  p = gsbn_fmac(p, t2, 1.0 / 355687428096000.0);  /*  1/17! */
  p = gsbn_fmac(p, t2, -1.0 / 1307674368000.0);   /* -1/15! */
  p = gsbn_fmac(p, t2, 1.0 / 6227020800.0);       /*  1/13! */
  p = gsbn_fmac(p, t2, -1.0 / 39916800.0);        /* -1/11! */
  p = gsbn_fmac(p, t2, 1.0 / 362880.0);           /*  1/9!  */
  p = gsbn_fmac(p, t2, -1.0 / 5040.0);            /* -1/7!  */
  p = gsbn_fmac(p, t2, 1.0 / 120.0);              /*  1/5!  */
  p = gsbn_fmac(p, t2, -1.0 / 6.0);               /* -1/3!  */
  return __builtin_fma(t * t2, p, t);
}

/* the float entry points by the short forms, the full sequences beyond their
 * range or guard */
GSBN_HD GSBN_INLINE float gsbn_expf_guarded(float x) {
  if (x >= -87.0f && x <= 88.0f) {
    const double y = gsbn_exp_short((double)x);
    if (gsbn_round_safe(y)) return (float)y;
  }
  return (float)gsbn_exp_cold((double)x);
}
GSBN_HD GSBN_INLINE float gsbn_logf_guarded(float x) {
  const uint32_t b = gsbn_fbits(x);
  if (b >= 0x00800000u && b < 0x7f800000u) { /* normal, positive, finite */
    const double y = gsbn_log_short(x);
    if (gsbn_round_safe(y)) return (float)y;
  }
  return (float)gsbn_log_cold((double)x);
}

/* The standard normal of two 24-bit words (gsbn_draw_unit) in double by the
 * short forms (k1 + 1 <= 2^24 is exact in float; cos(2 pi u) = sin(2 pi (1/4 -
 * a)) with a the distance of u from the nearest integer; the square root from
 * the seed and one Newton step) */
GSBN_HD GSBN_INLINE double gsbn_normal24_short(uint32_t k1, uint32_t k2) {
  const double t = -2.0 * gsbn_log_short((float)(k1 + 1u) * 5.9604644775390625e-08f);
  const double y = gsbn_rsq_seed(t);
  const double g = t * y;
  const double r = __builtin_fma(0.5 * g, __builtin_fma(-g, y, 1.0), g);
  const uint32_t a = k2 <= 0x800000u ? k2 : 0x1000000u - k2;
  return r * gsbn_sin2pi24(0x400000 - (int)a);
}

/* rounded, in full where the guard says so or u1 = 1 (whose result is a signed
 * zero) */
GSBN_HD GSBN_INLINE float gsbn_normal24_guarded(uint32_t k1, uint32_t k2) {
  const double z = gsbn_normal24_short(k1, k2);
  if (k1 != 0xffffffu && gsbn_round_safe(z)) return (float)z;
  return gsbn_normal24_cold(k1, k2);
}

/* gsbn_draw_unit */
GSBN_HD GSBN_INLINE void gsbn_draw_unit_guarded(uint64_t seed, uint32_t pop, uint32_t step,
                                                uint32_t unit, float* u01, float* z) {
  gsbn_u32x4 c;
  c.v[0] = unit;
  c.v[1] = step;
  c.v[2] = pop;
  c.v[3] = 0u;
  const gsbn_u32x4 w = gsbn_philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  *u01 = (float)(w.v[0] >> 8) * 5.9604644775390625e-08f; /* 2^-24 */
  *z = gsbn_normal24_guarded(w.v[1] >> 8, w.v[2] >> 8);
}

#endif /* GSBN_DETFAST_H */
