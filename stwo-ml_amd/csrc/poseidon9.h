// Poseidon hash of two felt252 (hades([a, b, 2])[0]) on the nine-limb
// device representation of felt9.h, for GPU Merkle trees.
//
// Same permutation as the host code (poseidon.h): 4 full rounds, 83 partial
// rounds with the compressed constants (one constant per partial round, the
// rest folded into the first of the last four full rounds), 4 full rounds;
// MDS [[3,1,1],[1,-1,1],[1,1,-2]].
//
// Full rounds are written as s0 = 3y0 + y1 + y2, s1 = y0 - y1 + y2,
// s2 = y0 + y1 - 2y2.  Partial rounds run on (u, w, x) = (s0 + s1, s0 - s1,
// s2): with y = x^3 and k the next partial constant,
//   u' = 2(u + w + y),  w' = 2u,  x' = u + k - 2y,
// which is the round s0' = 3s0 + s1 + y, s1' = s0 - s1 + y,
// s2' = s0 + s1 + k - 2y in sum/difference coordinates.  After the first
// partial round w = 2v with v the previous u, so a round is
//   u' = 2(2v + u) + Y,  v' = u,  x' = u + k - Y   with Y = 2y = x^2 * 2x,
// and s0 = u/2 + v, s1 = u/2 - v are recovered once after the last one.
//
// Value bounds (p ~ 2^251, R = 2^261): hash inputs below 8p; S-box inputs
// below 9p (full) and 8p (partial) give cubes below 1.1p; u is folded below
// 2^252 (1 + 2^-16) every partial round; outputs are normalized and below 5.2p.
#pragma once
#include "felt9.h"

namespace gkr {
namespace f9 {

struct hades_consts {
  fe first[4][3];  // rounds 0-3 (round 0, lane 2 unused: see y2_round0)
  fe y2_round0;    // (2 + first[0][2])^3: lane 2 of round 0 when the input lane 2 is 2
  fe partial0;     // constant added to lane 2 before partial round 0
  fe kd0;          // partial constant 1 plus kD4, for lane 2 after partial round 0
  fe u1;           // added to u after partial round 0 (see partial_u)
  fe ku[83];       // partial round r: added to u (ku[0] unused)
  uint32_t x6[83]; // partial round r: taken from limb 6 of x (signed; x6[0] unused)
  fe last[4][3];   // rounds 87-90, round 87 less what u and v still carry
};

GKR_HD void add(const fe& a, const fe& b, fe& r) {
#pragma unroll
  for (int k = 0; k < kLimbs; k++) r.l[k] = a.l[k] + b.l[k];
}

GKR_HD void full_linear(const fe& y0, const fe& y1, const fe& y2, fe& a, fe& b, fe& c) {
#pragma unroll
  for (int k = 0; k < kLimbs; k++) {
    const uint32_t d = consts::d4(k);
    a.l[k] = 3u * y0.l[k] + y1.l[k] + y2.l[k];
    b.l[k] = y0.l[k] + y2.l[k] + d - y1.l[k];
    c.l[k] = y0.l[k] + y1.l[k] + d - 2u * y2.l[k];
  }
  normalize(a);
  normalize(b);
  normalize(c);
}

template <typename K>
GKR_HD void full_round(fe& a, fe& b, fe& c, const K& rc0, const K& rc1, const K& rc2) {
  fe x0, x1, x2, y0, y1, y2;
  add(a, rc0, x0);
  add(b, rc1, x1);
  add(c, rc2, x2);
  cube(x0, y0);
  cube(x1, y1);
  cube(x2, y2);
  full_linear(y0, y1, y2, a, b, c);
}

// The round constants live in u: it is kept as U = u + g_r, where g_r is the
// constant that x' = u + g_r - Y needs up to a multiple of 2^174, so x' is one
// subtraction per limb.  With K_r = g_(r+1) - 2 g_r - 4 g_(r-1),
//   U' = 4V + 2U + Y + K_r,  V' = U,  x' = U - Y - x6 2^174,
// and K_r is the third addend of the carry pass's additions: it costs nothing.
// (Constants added to x, which was normalized: 328 VALU instructions a round
// instead of 301, seven weights of a Qwen2.5-14B layer 122.0 instead of 117.3 ms.)
//
// U' is folded to about [p, 2p) and normalized in the same pass: h p less one p
// is taken off, h = floor(U' / 2^251) up to the carries still to come, from the
// top limb before the carries.  h p only touches limbs 0, 6 and 8, and the one
// p's share of limbs 0 and 6 is part of ku.  Every limb sum has to stay in
// [0, 2^32): 4V + 2U + Y is at most 7 * 2^29 - 6 and the carry at most 7, so a
// ku limb is at most 2^29 - 8, and limbs 0 and 6 are at least 16 and 16 kP6
// (h <= 15).  x6, 0 or +-2^28, is there to move limb 6 into that range.
// (U, V normalized and below 2^252 (1 + 2^-16), Y above -p/16 and below 1.1p
// with limb 0 up to 2^29.)
GKR_HD void partial_u(const fe& u, const fe& v, const fe& Y, const fe& ku, fe& r) {
  uint32_t t[kLimbs];
#pragma unroll
  for (int k = 0; k < kLimbs; k++) t[k] = in_order((in_order((v.l[k] << 1) + u.l[k]) << 1) + Y.l[k]);  // two v_lshl_add
  const uint32_t top = t[8] + ku.l[8];
  const int32_t h = (int32_t)top >> 19;
  t[0] -= (uint32_t)h;
  t[6] -= (uint32_t)(h * (int32_t)kP6);
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint32_t x = t[k] + ku.l[k] + c;
    r.l[k] = x & kMask;
    c = x >> 29;
  }
  r.l[8] = ((top & (kP8 - 1u)) | kP8) + c;
}
// One partial round after the first: (u, v, x) -> (u', u, x'), u' in v; x has
// limbs of either sign, up to 2^29 (limb 6: 2^29 + 2^28) in magnitude, and a
// value between -1.2p and 7p.
GKR_HD void partial_round(const fe& u, fe& v, fe& x, const fe& ku, uint32_t x6) {
  fe d, x2, Y;
  twice(x, d);
  sqr2<true>(x, d, x2);
  mul<true>(x2, d, Y);
  partial_u(u, v, Y, ku, v);
#pragma unroll
  for (int k = 0; k < kLimbs; k++) x.l[k] = u.l[k] - Y.l[k] - (k == 6 ? x6 : 0u);
}

// out = hades([l, r, 2])[0]; l, r normalized, Montgomery, below 8p.
GKR_HD void hash2(const fe& l, const fe& r, const hades_consts& K, fe& out) {
  fe a, b, c;
  {
    fe x0, x1, y0, y1;
    add(l, K.first[0][0], x0);
    add(r, K.first[0][1], x1);
    cube(x0, y0);
    cube(x1, y1);
    full_linear(y0, y1, K.y2_round0, a, b, c);
  }
#pragma unroll 1
  for (int rr = 1; rr < 4; rr++) full_round(a, b, c, K.first[rr][0], K.first[rr][1], K.first[rr][2]);

  fe u, w, x;
#pragma unroll
  for (int k = 0; k < kLimbs; k++) {
    u.l[k] = a.l[k] + b.l[k];
    w.l[k] = a.l[k] + consts::d4(k) - b.l[k];
  }
  normalize(u);
  fold(u);
  normalize(w);
  add(c, K.partial0, x);
  fe v = u;
  {
    fe y;
    cube(x, y);
#pragma unroll
    for (int k = 0; k < kLimbs; k++) {
      const uint32_t un = u.l[k];
      u.l[k] = 2u * (un + w.l[k] + y.l[k]) + K.u1.l[k];
      x.l[k] = un + K.kd0.l[k] - 2u * y.l[k];
    }
    normalize(u);
    fold(u);
    normalize(x);
  }
#pragma unroll 1
  for (int r = 1; r < 83; r += 2) {  // the two halves exchange the roles of u and v: no copies
    partial_round(u, v, x, K.ku[r], K.x6[r]);
    partial_round(v, u, x, K.ku[r + 1], K.x6[r + 1]);
  }
#pragma unroll
  for (int k = 0; k < kLimbs; k++) c.l[k] = x.l[k] + consts::d4(k);
  normalize(c);
  halve(u);
#pragma unroll
  for (int k = 0; k < kLimbs; k++) {
    a.l[k] = u.l[k] + v.l[k];
    b.l[k] = u.l[k] + consts::d4(k) - v.l[k];
  }
  normalize(a);
  normalize(b);
#pragma unroll 1
  for (int rr = 0; rr < 3; rr++) full_round(a, b, c, K.last[rr][0], K.last[rr][1], K.last[rr][2]);
  {
    fe x0, x1, x2, y0, y1, y2;
    add(a, K.last[3][0], x0);
    add(b, K.last[3][1], x1);
    add(c, K.last[3][2], x2);
    cube(x0, y0);
    cube(x1, y1);
    cube(x2, y2);
#pragma unroll
    for (int k = 0; k < kLimbs; k++) out.l[k] = 3u * y0.l[k] + y1.l[k] + y2.l[k];
    normalize(out);
  }
}

}  // namespace f9
}  // namespace gkr
