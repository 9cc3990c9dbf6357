// The default moduli, and the exact combine of 12 to 15 of them by remainder
// weights (host and device: the CPU tests run what the kernels run).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "fp64emu.h"

namespace {

constexpr int kMaxP = FP64EMU_MAXP;
// x + kMagic (|x| < 2^51) lands on the integer grid of [2^52, 2^53): the sum
// rounds x to the nearest integer, ties to even.
constexpr double kMagic = 6755399441055744.0;

typedef __int128 i128;

__host__ __device__ constexpr int inv_mod(int a, int m) {
  // Extended Euclid on (a mod m, m); m <= 256, gcd 1 by coprimality.
  int r0 = ((a % m) + m) % m, r1 = m, s0 = 1, s1 = 0;
  while (r1 != 0) {
    const int q = r0 / r1;
    int t = r0 - q * r1; r0 = r1; r1 = t;
    t = s0 - q * s1; s0 = s1; s1 = t;
  }
  return ((s0 % m) + m) % m;
}

// The reference's modulus list (fp64_emu/__init__.py:20-22), every plan a
// prefix of it: the modulus-count-specialised reconstruction takes its
// constants from this table at compile time.
constexpr int kDefaultModuli[kMaxP] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227,
                                       223, 217, 211, 199, 197, 193, 191, 181, 179, 173};

// The default list's Chinese remainder weights, for the exact combine: with
// W_t = (M / p_t) ((M / p_t)^-1 mod p_t) taken mod M in (-M/2, M/2], the
// product is X = sum_t r_t W_t - q M for any residues r_t, q the nearest
// integer to the sum over M.  W_t and M are cut into three slices of kCrtBits
// bits (balanced, but for the top one), so that each slice's sum over
// residues (or sums of a K-split's residues: crt_exact) is an exact float64
// integer:  sum_t r_t W_t = s1 4^kCrtBits + s2 2^kCrtBits + s3.
// The digits' serial chain, their 14-step Horner and the 128-bit combine took
// 190 vector instructions an element at 14 moduli, this 120 with no serial
// part, and a K-split's sums need no reduction first.  Whole calls against the
// digits: 128 x 128 x 4096 (8 splits) 43.2 -> 41.3 us, 64 x 512^3 487.6 ->
// 482.3 us, 1024^3 62.0 -> 60.6 us; from 4096^3 on even (the reconstruction
// there streams 18 bytes in and 8 out an element at 5.5 TB/s either way).
constexpr int kCrtBits = 39;

struct CrtTab {
  double w[3][kMaxP];   // slices of W_t, the top one first
  double m[3];          // slices of M
  double inv;           // 2^kCrtBits / M
  double top;           // the largest |s| of any slice, before and after q M, at |r_t| <= p_t / 2
};

__host__ __device__ constexpr void crt_slices(i128 v, double (&out)[3]) {
  for (int i = 2; i >= 1; --i) {
    const i128 half = (i128)1 << (kCrtBits - 1);
    const i128 low = ((v + half) & (((i128)1 << kCrtBits) - 1)) - half;
    out[i] = (double)(long long)low;
    v = (v - low) >> kCrtBits;
  }
  out[0] = (double)(long long)v;
}

__host__ __device__ constexpr CrtTab crt_tables(int P) {
  CrtTab T{};
  i128 M = 1;
  for (int t = 0; t < P; ++t) M *= kDefaultModuli[t];
  double sums[3] = {0.0, 0.0, 0.0}, all = 0.0;
  for (int t = 0; t < P; ++t) {
    const int p = kDefaultModuli[t];
    const i128 N = M / p;
    i128 W = N * inv_mod((int)(N % p), p);
    if (2 * W > M) W -= M;
    double s[3] = {};
    crt_slices(W, s);
    for (int i = 0; i < 3; ++i) {
      T.w[i][t] = s[i];
      sums[i] += (double)(p / 2) * (s[i] < 0 ? -s[i] : s[i]);
    }
    all += (double)(p / 2) * (double)(W < 0 ? -W : W);
  }
  crt_slices(M, T.m);
  T.inv = (double)(1ll << kCrtBits) / (double)M;
  for (int i = 0; i < 3; ++i) {
    const double v = sums[i] + (all / (double)M + 1.0) * (T.m[i] < 0 ? -T.m[i] : T.m[i]);
    T.top = v > T.top ? v : T.top;
  }
  return T;
}

// Modulus counts whose sums of residues |r_t| <= 128 fold stay exact.
__host__ __device__ constexpr bool crt_exact(int P, int fold) {
  if (P < 12 || P > 15) return false;
  return crt_tables(P).top * fold < 9007199254740992.0;   // 2^53
}

// RN(X + cv 2^cshift) 2^sh for the slice sums s1, s2, s3 of an element (before
// the multiple of M comes off): exactly rounded, as the 128-bit combine.  Every
// value is an integer, and each Fast2Sum's first operand a multiple of the
// second one's ulp (a slice of weight 2^39 against at most 52 bits below 2^91,
// and so on), which makes its error exact whichever operand is larger.
template <int kP>
__host__ __device__ __forceinline__ double crt_combine(double s1, double s2, double s3, const double cv,
                                                       const int cshift, const int sh) {
  constexpr CrtTab T = crt_tables(kP);
  constexpr double kB = (double)(1ll << kCrtBits);
  // The nearest integer to the sum over M, from the sum's top 53 bits: off
  // only within 2^-40 of a tie, while the width pick keeps |X| below 0.36 M.
  const double q = fma(fma(s1, kB, s2), T.inv, kMagic) - kMagic;
  s1 = fma(-q, T.m[0], s1);
  s2 = fma(-q, T.m[1], s2);
  s3 = fma(-q, T.m[2], s3);
  // (h, l) = s1 2^39 + s2, in units of 2^39.
  const double h = fma(s1, kB, s2);
  const double l = s2 - fma(s1, -kB, h);
  // (u, v) = the correction + s3.
  const double d = ldexp(cv, cshift);
  const double u = d + s3;
  const double v = s3 - (u - d);
  // (p, e) = l + u, (h2, p2) = h + p: the value is h2 + p2 + (e + v).
  const double p = fma(l, kB, u);
  const double e = u - fma(l, -kB, p);
  const double h2 = fma(h, kB, p);
  const double p2 = p - fma(h, -kB, h2);
  // p2 + (e + v) rounded to odd (its last bit set when inexact), so that the
  // last addition rounds once: it is inexact only beyond 2^53, when h2 is
  // beyond 2^105 and its rounding position far above that bit.
  const double s = e + v;
  const double y = p2 + s;
  const double err = s - (y - p2);
  uint64_t yb;
  __builtin_memcpy(&yb, &y, 8);
  uint64_t eb;
  __builtin_memcpy(&eb, &err, 8);
  const bool inexact = err != 0.0;
  const int64_t opposite = (int64_t)(eb ^ yb) >> 63;   // -1: |y| is above the exact magnitude
  yb = inexact ? (yb + (uint64_t)opposite) | 1u : yb;
  double yo;
  __builtin_memcpy(&yo, &yb, 8);
  return ldexp(h2 + yo, sh);
}

// kE elements' values from their residues r(t, e) (any representatives, or
// sums of representatives: crt_exact), correction sums cv and shifts.
template <int kP, int kE, typename R>
__host__ __device__ __forceinline__ void crt_values(const R& r, const double (&cv)[kE], const int cshift,
                                           const int (&sh)[kE], double (&val)[kE]) {
  constexpr CrtTab T = crt_tables(kP);
  double s1[kE] = {}, s2[kE] = {}, s3[kE] = {};
#pragma unroll
  for (int t = 0; t < kP; ++t)
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      const double d = (double)r(t, e);
      s1[e] = fma(d, T.w[0][t], s1[e]);
      s2[e] = fma(d, T.w[1][t], s2[e]);
      s3[e] = fma(d, T.w[2][t], s3[e]);
    }
#pragma unroll
  for (int e = 0; e < kE; ++e) val[e] = crt_combine<kP>(s1[e], s2[e], s3[e], cv[e], cshift, sh[e]);
}

}  // namespace
