/*
 * mc_fx.h -- the exact fixed-point arithmetic of the tallies: conversion of
 * a double term to a signed 128-bit integer with 2^-88 resolution and the
 * correctly rounded conversion of a 128-bit sum back to double.
 *
 * Integer code only (plus one ldexp), so it compiles as HIP device code and
 * as plain host C/C++ (gcc) for CPU-side tests; the device kernels use this
 * exact source.
 */
#ifndef MC_FX_H
#define MC_FX_H

#include <stdint.h>

#include "mc_math.h" /* mc_asu64, MC_FN, MC_FN_COLD */

#if defined(__HIPCC__)
#define MC_FN_HD __host__ __device__ __forceinline__ static
#else
#define MC_FN_HD static inline
#endif

/* ------------------------------------------------- exact fixed-point tally
 * A term v maps to the signed 128-bit integer round_half_up(v * 2^88),
 * stored as (lo, hi) two's complement.  Non-finite terms and |v| >= 2^39 set
 * flag bits instead (1 NaN, 2 +inf, 4 -inf, 8 out of range).  Integer sums
 * are exact, so the tally does not depend on the order in which lanes, waves
 * and blocks add their terms. */
#define MC_FX_FRAC 88

typedef struct mc_fx {
  uint64_t lo;
  uint64_t hi;
} mc_fx;

/* The conversion for every term (zero, subnormal, negative, large and
   non-finite ones included), with its flags. */
typedef struct mc_fx_flagged {
  mc_fx v;
  uint32_t flags;
} mc_fx_flagged;

MC_FN_COLD mc_fx_flagged mc_fx_from_double_general(double v) {
  mc_fx_flagged out;
  out.flags = 0;
  uint64_t b = mc_asu64(v);
  uint32_t E = (uint32_t)(b >> 52) & 0x7FFu;
  mc_fx r = {0, 0};
  out.v = r;
  if (E == 0x7FFu) {
    out.flags = (b & 0x000FFFFFFFFFFFFFULL) ? 1u : ((b >> 63) ? 4u : 2u);
    return out;
  }
  if (E >= 1023u + 39u) {
    out.flags = 8u;
    return out;
  }
  if (E == 0u) return out; /* zero or subnormal: below 2^-89 -> 0 */
  uint64_t M = (b & 0x000FFFFFFFFFFFFFULL) | 0x0010000000000000ULL;
  int s = (int)E - 987; /* v = M * 2^(E-1075); v*2^88 = M * 2^(E-987) */
  if (s >= 64) {
    r.hi = M << (s - 64);
  } else if (s > 0) {
    r.lo = M << s;
    r.hi = M >> (64 - s);
  } else if (s == 0) {
    r.lo = M;
  } else if (s > -64) {
    r.lo = ((M >> (-s - 1)) + 1) >> 1; /* round half up */
  }
  if (b >> 63) { /* negate (two's complement) */
    r.lo = ~r.lo + 1;
    r.hi = ~r.hi + (r.lo == 0 ? 1 : 0);
  }
  out.v = r;
  return out;
}

/* Fast path for 2^-35 <= |v| < 2^28: |v| * 2^88 = M * 2^s with 0 < s < 64,
   so the 128-bit integer is two shifts of the 53-bit significand (negated for
   v < 0), exactly as in the general path.  Returns 0 and leaves r alone
   outside that range.  POSITIVE_ONLY sends negative terms to the general
   path too (the transport's deposits are never negative; the adjoint's terms
   are). */
#define MC_FX_FAST(POSITIVE_ONLY, v, r, taken)                               \
  do {                                                                      \
    const uint64_t b_ = mc_asu64(v);                                        \
    const int s_ = (POSITIVE_ONLY) ? (int)((uint32_t)(b_ >> 52)) - 987      \
                                   : (int)((uint32_t)(b_ >> 52) & 0x7FFu) - 987; \
    (taken) = (unsigned)(s_ - 1) < 63u;                                     \
    if (taken) {                                                            \
      const uint64_t M_ = (b_ & 0x000FFFFFFFFFFFFFULL) | 0x0010000000000000ULL; \
      (r).lo = M_ << s_;                                                    \
      (r).hi = M_ >> (64 - s_);                                             \
      if (!(POSITIVE_ONLY) && (b_ >> 63)) { /* two's complement */          \
        (r).lo = ~(r).lo + 1;                                               \
        (r).hi = ~(r).hi + ((r).lo == 0 ? 1 : 0);                           \
      }                                                                     \
    }                                                                       \
  } while (0)

/* round_half_up(v * 2^88) as a signed 128-bit integer; flags as above.
   positive_only selects the fast path's sign handling (results identical). */
MC_FN mc_fx mc_fx_from_double_p(double v, uint32_t *flags, int positive_only) {
  mc_fx r;
  int taken;
  if (positive_only) {
    MC_FX_FAST(1, v, r, taken);
  } else {
    MC_FX_FAST(0, v, r, taken);
  }
  if (taken) return r;
  const mc_fx_flagged g = mc_fx_from_double_general(v);
  *flags |= g.flags;
  return g.v;
}

MC_FN mc_fx mc_fx_from_double(double v, uint32_t *flags) {
  return mc_fx_from_double_p(v, flags, 0);
}

/* Correctly rounded conversion of the 128-bit sum back to double. */
MC_FN_HD double mc_fx_to_double(uint64_t lo, uint64_t hi) {
  int neg = (int64_t)hi < 0;
  if (neg) {
    lo = ~lo + 1;
    hi = ~hi + (lo == 0 ? 1 : 0);
  }
  double d;
  if (hi == 0) {
    d = (double)lo * 0x1p-88;
  } else {
    int lz = __builtin_clzll(hi);
    uint64_t top = lz ? ((hi << lz) | (lo >> (64 - lz))) : hi;
    uint64_t rest = lz ? (lo << lz) : lo;
    top |= (rest != 0) ? 1u : 0u; /* sticky bit below the rounding position */
    d = __builtin_ldexp((double)top, 64 - lz - MC_FX_FRAC);
  }
  return neg ? -d : d;
}

MC_FN_HD double mc_fx_finalize(uint64_t lo, uint64_t hi, uint32_t flags) {
  if ((flags & 1u) || (flags & 8u) || ((flags & 6u) == 6u)) return __builtin_nan("");
  if (flags & 2u) return __builtin_inf();
  if (flags & 4u) return -__builtin_inf();
  return mc_fx_to_double(lo, hi);
}

/* ------------------------------------------------------- two-limb tallies
   A block's tally in LDS keeps two 64-bit sums per cell that never carry into
   each other: for a term v, limb 1 takes n1 = v rounded to a multiple of
   2^(L-88) and limb 0 the signed rest in units of 2^-88, so that
   n1 * 2^L + n0 is the term's fixed-point integer exactly.  No add needs the
   other limb's result, so both are plain atomic adds without a returned
   value.  |n0| <= 2^(L-1); with 0 <= v < 2^V, n1 <= 2^(V+88-L).  After N
   terms limb 0 stays within a signed and limb 1 within an unsigned 64-bit
   word while N <= 2^(64-L) and N <= 2^(L-V-24); L = 44 + floor(V/2) makes
   the two bounds (nearly) equal.  A block moves its limbs to the global
   128-bit tally (mc_fx_limbs) before N terms can have been added to a cell.
   Both limbs come from adding constants whose ulp is the limb's unit:
   c1 = 1.5 * 2^(L-36), 1.5 * 2^-36. */
typedef struct {
  double c1;
  uint32_t c1_hi;  /* high word of c1 (its low word is zero) */
  uint32_t range;  /* high word of 2^V less that of 2^-36 */
  int L;
} mc_fx_split;

#define MC_FX_C2 0x1.8p-36
#define MC_FX_C2_HI ((uint32_t)((1023 - 36) << 20 | 0x80000))
#define MC_FX_HI36 ((uint32_t)((1023 - 36) << 20)) /* high word of 2^-36 */
#define MC_FX_HI88 ((uint32_t)((1023 - 88) << 20)) /* high word of 2^-88 */

/* terms below 2^V, -35 <= V <= 14: v + c1 stays in c1's binade while
   2^V <= c1 / 3, which fails at V = 15 */
MC_FN_HD mc_fx_split mc_fx_split_for(int V) {
  mc_fx_split S;
  S.L = 44 + (V >> 1);
  S.c1_hi = (uint32_t)((1023 + S.L - 36) << 20 | 0x80000);
  const uint64_t b = (uint64_t)S.c1_hi << 32;
  __builtin_memcpy(&S.c1, &b, 8);
  S.range = ((uint32_t)(1023 + V) << 20) - MC_FX_HI36;
  return S;
}

/* log2 of the number of terms a cell may take between two moves */
MC_FN_HD int mc_fx_split_log2_terms(int V) {
  const int L = 44 + (V >> 1);
  return 64 - L < L - V - 24 ? 64 - L : L - V - 24;
}

/* v in [2^-36, 2^V): its unit 2^-88 or coarser, no rounding */
MC_FN_HD int mc_fx_split_direct(double v, const mc_fx_split *S) {
  uint64_t b;
  __builtin_memcpy(&b, &v, 8);
  return (uint32_t)(b >> 32) - MC_FX_HI36 < S->range;
}

/* v = 0 or in [2^-88, 2^-36): rounded half up to a multiple of 2^-88 (then as
   mc_fx_split_direct).  v * 2^88 + 1/2 in one fma: exact, or (across a power
   of two) rounded without crossing an integer.  Other terms return 0. */
MC_FN_HD int mc_fx_split_small(double *v) {
  uint64_t b;
  __builtin_memcpy(&b, v, 8);
  const uint32_t h = (uint32_t)(b >> 32);
  if (!(h - MC_FX_HI88 < MC_FX_HI36 - MC_FX_HI88 || b == 0)) return 0;
  *v = __builtin_floor(__builtin_fma(*v, 0x1p88, 0.5)) * 0x1p-88;
  return 1;
}

/* v in [0, 2^-88): rounded half up to 0 or 2^-88.  Other terms return 0. */
MC_FN_HD int mc_fx_split_tiny(double *v) {
  uint64_t b;
  __builtin_memcpy(&b, v, 8);
  if ((uint32_t)(b >> 32) >= MC_FX_HI88) return 0;
  *v = *v < 0x1p-89 ? 0.0 : 0x1p-88;
  return 1;
}

/* the limbs of a term that one of the three accepts */
MC_FN_HD void mc_fx_split_limbs(double v, const mc_fx_split *S, uint64_t *n0, uint64_t *n1) {
  const double h = v + S->c1;
  const double rest = v - (h - S->c1);
  const double l = rest + MC_FX_C2;
  uint64_t hb, lb;
  __builtin_memcpy(&hb, &h, 8);
  __builtin_memcpy(&lb, &l, 8);
  *n1 = (uint64_t)((uint32_t)(hb >> 32) - S->c1_hi) << 32 | (uint32_t)hb;
  *n0 = (uint64_t)((uint32_t)(lb >> 32) - MC_FX_C2_HI) << 32 | (uint32_t)lb;
}

/* n1 * 2^L + n0 as the 128-bit integer (n0 signed, n1 unsigned) */
MC_FN_HD mc_fx mc_fx_limbs(uint64_t n0, uint64_t n1, int L) {
  mc_fx r;
  r.lo = (n1 << L) + n0;
  r.hi = (n1 >> (64 - L)) + (uint64_t)((int64_t)n0 >> 63) + (r.lo < n0 ? 1u : 0u);
  return r;
}

/* Terms of either sign (the gradients'): |v| < 2^V, limb 1 signed, so half as
   many terms.  Rounding as in mc_fx_from_double_general: the magnitude half
   up.  (Most terms are zero: callers skip those before the test.) */
MC_FN_HD int mc_fx_split_signed_log2_terms(int V) {
  const int L = 44 + (V >> 1);
  return 64 - L < L - V - 25 ? 64 - L : L - V - 25;
}

MC_FN_HD int mc_fx_split_signed_direct(double v, const mc_fx_split *S) {
  uint64_t b;
  __builtin_memcpy(&b, &v, 8);
  return ((uint32_t)(b >> 32) & 0x7FFFFFFFu) - MC_FX_HI36 < S->range;
}

MC_FN_HD int mc_fx_split_signed_small(double *v) {
  double a = __builtin_fabs(*v);
  if (!mc_fx_split_small(&a)) return 0;
  *v = __builtin_copysign(a, *v);
  return 1;
}

MC_FN_HD int mc_fx_split_signed_tiny(double *v) {
  double a = __builtin_fabs(*v);
  if (!mc_fx_split_tiny(&a)) return 0;
  *v = __builtin_copysign(a, *v);
  return 1;
}

MC_FN_HD mc_fx mc_fx_signed_limbs(uint64_t n0, uint64_t n1, int L) {
  mc_fx r;
  r.lo = (n1 << L) + n0;
  r.hi = (uint64_t)((int64_t)n1 >> (64 - L)) + (uint64_t)((int64_t)n0 >> 63) +
         (r.lo < n0 ? 1u : 0u);
  return r;
}

#endif /* MC_FX_H */
