// felt252 arithmetic for GPU lanes: p = 2^251 + 17*2^192 + 1 held in nine
// 29-bit limbs (261 bits), Montgomery form with R = 2^261.
//
// Why 29 bits: a product of two limbs below 2^30 is below 2^60, so a column
// of at most nine such products plus the reduction terms stays below 2^64.
// Every partial product is then one v_mad_u64_u32 into a 64-bit column
// accumulator with no carry handling; carries are resolved once, during the
// reduction.  The prime has three non-zero limbs (limb 0 = 1, limb 6 =
// 17*2^18, limb 8 = 2^19) and -p^-1 = -1 mod 2^29, so each of the nine
// Montgomery digits is the negated low limb of its column and costs two mads.
//
// Representation rules (all values are representatives, not canonical):
//   normalized: limbs in [0, 2^29), value below 2^261;
//   mul/sqr inputs: limbs below 2^30 (the sum of two normalized values is
//     fine), output normalized with value < p + a*b/R; their signed forms take
//     limbs of either sign (a difference of two normalized values), and their
//     output's top limb has the sign of the value;
//   the linear layer adds limb-wise and subtracts through kD4, a
//     representation of 4p whose limbs dominate any normalized subtrahend
//     below 1.1p (limbs 0-7 at least 2^30 - 2, limb 8 at least 2^21 - 2).
// Functions are __host__ __device__ so the same code runs in CPU tests.
#pragma once
#include <stdint.h>

#ifndef GKR_HD
#if defined(__HIPCC__)
#define GKR_HD __host__ __device__ __forceinline__
#else
#define GKR_HD inline
#endif
#endif

namespace gkr {
namespace f9 {

constexpr int kLimbs = 9;
constexpr uint32_t kMask = (1u << 29) - 1;
constexpr uint32_t kP6 = 17u << 18;  // limb 6 of p
constexpr uint32_t kP8 = 1u << 19;   // limb 8 of p

struct fe {
  uint32_t l[kLimbs];
};

// kD4: 4p = 2^253 + 68*2^192 + 4 with 2^30 moved from each limb i+1 into limb i
// (adds 2^30 to limb i and subtracts 2 from limb i+1, value unchanged).
struct consts {
  static constexpr uint32_t d4(int i) {
    return i == 0 ? 4u + (1u << 30)
           : i == 6 ? (68u << 18) + (1u << 30) - 2u
           : i == 8 ? (1u << 21) - 2u
                    : (1u << 30) - 2u;
  }
};

// Hides a constant from the optimizer, so that it stays a multiplier of
// v_mad_u64_u32 instead of being rewritten as separate shifts/adds.
template <typename T>
GKR_HD T opaque(T v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(v));
#endif
  return v;
}
// The same for a per-lane value: keeps sums in the written order.
template <typename T>
GKR_HD T in_order(T v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(v));
#endif
  return v;
}

// Products are scanned column by column (column k collects the products of
// limbs i and k - i): one 64-bit accumulator runs through all columns, so the
// carry from column k is the addend of column k + 1's first v_mad_u64_u32 and
// costs no addition of its own.  Column k < 9 ends with the reduction digit
// m_k = -(acc + e) mod 2^29, e being the 1 the digits below have carried in:
// m_0 = 2^29 - (acc mod 2^29), and from column 1 on, where the low columns
// always carry 1 more than acc >> 29 holds, m_k = 2^29 - 1 - (acc mod 2^29),
// one v_bfi.  m_k enters columns k + 6 and k + 8 (limbs 6 and 8 of p; limb 0
// cancels the column).  The carried 1 arrives in column 9, so it is added to
// limb 0 of the result.  The sum of the m's is at most 2^261, so the result is
// below p + t / 2^261; limb 0 is at most 2^29, the others below 2^29.
//
// Digits and carries are the same in two's complement, so limbs of either sign
// (S) only need the signed mad and the arithmetic shift.
//
// Per product 81 (or 45 in a square) + 18 v_mad_u64_u32, 16 shifts and about 20
// 32-bit operations.  k_merkle_level is bound by VALU issue, most of it the
// mads.  Against unordered columns with the exact digit 2^29 - (t mod 2^29)
// (two more operations a digit, a 64-bit addition per carry) and a partial
// round that folded and normalized u in two passes: a partial round 333
// instead of about 430 VALU instructions, the 275 M hashes of seven weights
// of a Qwen2.5-14B layer 307.8 -> 243.5 ms (0.89 -> 1.13 G hashes/s).  Every
// sum is kept in the written order (in_order): left to itself the compiler
// adds a column's products first and the carry with a separate 64-bit
// addition (262.8 ms).
struct columns {
  uint64_t acc;
  uint32_t m[9];
  uint32_t p6, p8;
};
GKR_HD void column_begin(columns& c) {
  c.acc = 0;
  c.p6 = opaque(kP6);
  c.p8 = opaque(kP8);
}
// a * b of limbs (S: signed)
template <bool S>
GKR_HD uint64_t limb_mul(uint32_t a, uint32_t b) {
  if constexpr (S) return (uint64_t)((int64_t)(int32_t)a * (int32_t)b);
  return (uint64_t)a * b;
}
// the reduction terms and the digit (or result limb) of column k, after its products
template <bool S, int K>
GKR_HD void column_end(columns& c, fe& r) {
  if constexpr (K >= 6 && K < 15) c.acc = in_order(c.acc + (uint64_t)c.m[K - 6] * c.p6);
  if constexpr (K >= 8) c.acc = in_order(c.acc + (uint64_t)c.m[K - 8] * c.p8);
  if constexpr (K < 9)
    c.m[K] = (~(uint32_t)c.acc & kMask) + (K == 0 ? 1u : 0u);
  else
    r.l[K - 9] = ((uint32_t)c.acc & kMask) + (K == 9 ? 1u : 0u);
  if constexpr (S)
    c.acc = (uint64_t)((int64_t)c.acc >> 29);
  else
    c.acc >>= 29;
}

template <bool S, int K>
GKR_HD void mul_columns(const fe& a, const fe& b, columns& c, fe& r) {
  constexpr int I0 = K > 8 ? K - 8 : 0;
  c.acc = in_order(c.acc + limb_mul<S>(a.l[I0], b.l[K - I0]));  // the carry is this mad's addend
#pragma unroll
  for (int i = I0 + 1; i <= (K < 8 ? K : 8); i++) c.acc = in_order(c.acc + limb_mul<S>(a.l[i], b.l[K - i]));
  column_end<S, K>(c, r);
  if constexpr (K < 16) mul_columns<S, K + 1>(a, b, c, r);
}
// Inputs: limbs whose pairwise products sum below 2^64 - 2^52 in every column
// (limbs below 2^30 on both sides with top limbs below 2^29, or a normalized
// value by limbs below 2^31).  S: sums within +-(2^63 - 2^52).
template <bool S = false>
GKR_HD void mul(const fe& a, const fe& b, fe& r) {
  columns c;
  fe o;
  column_begin(c);
  mul_columns<S, 0>(a, b, c, o);
  o.l[8] = (uint32_t)c.acc;
  r = o;
}

template <bool S, int K>
GKR_HD void sqr_columns(const fe& a, const fe& d, columns& c, fe& r) {
  constexpr int I0 = K > 8 ? K - 8 : 0;
  c.acc = in_order(c.acc + limb_mul<S>(a.l[I0], 2 * I0 < K ? d.l[K - I0] : a.l[I0]));
#pragma unroll
  for (int i = I0 + 1; 2 * i < K; i++) c.acc = in_order(c.acc + limb_mul<S>(a.l[i], d.l[K - i]));
  if constexpr (K % 2 == 0 && 2 * I0 < K) c.acc = in_order(c.acc + limb_mul<S>(a.l[K / 2], a.l[K / 2]));
  column_end<S, K>(c, r);
  if constexpr (K < 16) sqr_columns<S, K + 1>(a, d, c, r);
}
// a^2 with d = 2a limb by limb (off-diagonal products taken once against d).
template <bool S = false>
GKR_HD void sqr2(const fe& a, const fe& d, fe& r) {
  columns c;
  fe o;
  column_begin(c);
  sqr_columns<S, 0>(a, d, c, o);
  o.l[8] = (uint32_t)c.acc;
  r = o;
}
GKR_HD void twice(const fe& a, fe& d) {
#pragma unroll
  for (int i = 0; i < kLimbs; i++) d.l[i] = a.l[i] << 1;
}
GKR_HD void sqr(const fe& a, fe& r) {
  fe d;
  twice(a, d);
  sqr2(a, d, r);
}

// x^3
GKR_HD void cube(const fe& x, fe& r) {
  fe x2;
  sqr(x, x2);
  mul(x2, x, r);
}

// Carry propagation of non-negative limbs below 2^32; value must be below 2^261.
GKR_HD void normalize(fe& a) {
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint32_t v = a.l[k] + c;  // a.l[k] < 2^32 - 8 and c < 8 in every caller
    a.l[k] = v & kMask;
    c = v >> 29;
  }
  a.l[8] += c;
}

// Signed carry propagation (limbs read as int32); value must be in [0, 2^261).
GKR_HD void normalize_signed(fe& a) {
  int32_t c = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int32_t v = (int32_t)a.l[k] + c;
    a.l[k] = (uint32_t)v & kMask;
    c = v >> 29;  // arithmetic shift
  }
  a.l[8] = (uint32_t)((int32_t)a.l[8] + c);
}

// Normalized a -> normalized value congruent mod p and below 2^252: with
// h = a >> 251, subtract max(h - 1, 0) * p.
// Requires h < 2^7 (value below 2^258) so the limb 6 adjustment fits.
GKR_HD void fold(fe& a) {
  const int32_t h = (int32_t)(a.l[8] >> 19);
  const int32_t k = h > 0 ? h - 1 : 0;
  a.l[8] -= (uint32_t)k << 19;
  a.l[6] = (uint32_t)((int32_t)a.l[6] - k * (int32_t)kP6);
  a.l[0] = (uint32_t)((int32_t)a.l[0] - k);
  normalize_signed(a);
}

// a / 2 mod p for normalized a: add p when odd, then shift right by one bit.
// Output limbs below 2^29 + 2^28.
GKR_HD void halve(fe& a) {
  const uint32_t odd = a.l[0] & 1u;
  a.l[0] += odd;
  a.l[6] += odd * kP6;
  a.l[8] += odd * kP8;
#pragma unroll
  for (int k = 0; k < 8; k++) a.l[k] = (a.l[k] >> 1) + ((a.l[k + 1] & 1u) << 28);
  a.l[8] >>= 1;
}

// Canonical 256-bit little-endian words <-> limbs (no Montgomery conversion).
GKR_HD void from_words(const uint32_t w[8], fe& r) {
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const int bit = 29 * k, wi = bit >> 5, off = bit & 31;
    uint64_t v = (uint64_t)w[wi] >> off;
    if (wi + 1 < 8) v |= (uint64_t)w[wi + 1] << (32 - off);
    r.l[k] = (uint32_t)v & kMask;
  }
}
GKR_HD void to_words(const fe& a, uint32_t w[8]) {
  uint64_t acc = 0;
  int have = 0, k = 0;
#pragma unroll
  for (int wi = 0; wi < 8; wi++) {
    while (have < 32 && k < 9) {
      acc |= (uint64_t)a.l[k++] << have;
      have += 29;
    }
    w[wi] = (uint32_t)acc;
    acc >>= 32;
    have -= 32;
  }
}

// Value in [0, 2^253), limb 0 up to 2^29 -> canonical residue in [0, p).
GKR_HD void canonicalize(fe& a) {
  normalize(a);
  // subtract p up to 4 times (value < 2^253 < 5p)
#pragma unroll
  for (int rep = 0; rep < 4; rep++) {
    fe d;
    int32_t c = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const uint32_t pk = k == 0 ? 1u : k == 6 ? kP6 : k == 8 ? kP8 : 0u;
      int32_t v = (int32_t)a.l[k] - (int32_t)pk + c;
      c = v >> 29;
      d.l[k] = k < 8 ? ((uint32_t)v & kMask) : (uint32_t)v;
    }
    if ((int32_t)d.l[8] >= 0) a = d;
  }
}

}  // namespace f9
}  // namespace gkr
