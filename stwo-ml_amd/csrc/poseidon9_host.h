// Host-side set-up for the device Poseidon (poseidon9.h): round constants and
// Montgomery conversion constants in the nine-limb, R = 2^261 representation,
// derived from the host permutation's compressed constants (poseidon.h).
#pragma once
#include "poseidon.h"
#include "poseidon9.h"

namespace gkr {
namespace f9 {

// Canonical integer below p -> limbs (no Montgomery conversion).
inline fe from_canonical(const felt& canon) {
  uint32_t w[8];
  felt_canon_to_words(canon, w);
  fe r;
  from_words(w, r);
  return r;
}

// Host Montgomery form (x * 2^256 mod p) -> device Montgomery form (x * 2^261 mod p).
inline felt raw(const felt& m) {  // as an integer below p
  felt v = m;
  for (int i = 0; i < 5; i++) v = felt_add(v, v);
  return v;
}
inline fe from_host_mont(const felt& m) { return from_canonical(raw(m)); }

struct setup {
  hades_consts k;
  fe r2;   // 2^522 mod p: mul(x, r2) takes a canonical x to Montgomery form
  fe one;  // plain 1: mul(x, one) takes Montgomery form back to a representative of x
  // ku and x6 (see partial_u) from the constants x needs; what u and v carry
  // after the last partial round comes off round 87's constants.
  void partial_constants(const hades_rc& h) {
    const felt zero{{0, 0, 0, 0}}, unit{{0, 0, 0, 1ull << 10}}, half_unit{{0, 0, 0, 1ull << 9}};  // 2^28, 2^27 at limb 6
    felt g0 = zero, g1 = raw(h.partial[2]);
    k.u1 = from_canonical(g1);
    k.ku[0] = fe{};
    k.x6[0] = k.x6[1] = 0;
    int shift = 0, shift_before = 0;  // x6 of rounds r + 1 and r, in units of 2^28
    for (int r = 1; r < 83; r++) {
      felt g2 = r + 2 < 83 ? raw(h.partial[r + 2]) : zero;
      const felt g01 = felt_add(felt_add(g0, g0), g1);
      const felt base = felt_sub(g2, felt_add(g01, g01));
      shift_before = shift;
      shift = 0;
      const uint32_t l6 = from_canonical(base).l[6] + kP6;
      if (l6 < 16 * kP6)
        shift = 1;
      else if (l6 > kMask - 7)
        shift = -1;
      const felt add = shift > 0 ? unit : shift < 0 ? felt_sub(zero, unit) : zero;
      k.ku[r] = from_canonical(felt_add(base, add));
      k.ku[r].l[0] += 1;
      k.ku[r].l[6] += kP6;
      if (r < 82) k.x6[r + 1] = (uint32_t)(shift * (1 << 28));
      g0 = g1;
      g1 = felt_add(g2, add);
    }
    // u = U - shift 2^28, v = V - shift_before 2^28 (at limb 6); s0 = u / 2 + v, s1 = u / 2 - v
    felt d0 = zero, d1 = zero;
    auto off = [](felt& d, int s, const felt& by) { d = s > 0 ? felt_sub(d, by) : s < 0 ? felt_add(d, by) : d; };
    off(d0, shift, half_unit);
    off(d1, shift, half_unit);
    off(d0, shift_before, unit);
    off(d1, -shift_before, unit);
    k.last[0][0] = from_canonical(felt_add(raw(h.full_last[0][0]), d0));
    k.last[0][1] = from_canonical(felt_add(raw(h.full_last[0][1]), d1));
  }
  setup() {
    const hades_rc& h = hades_constants();
    for (int r = 0; r < 4; r++)
      for (int j = 0; j < 3; j++) {
        k.first[r][j] = from_host_mont(h.full_first[r][j]);
        k.last[r][j] = from_host_mont(h.full_last[r][j]);
      }
    fe x2;
    add(from_host_mont(felt_from_u64(2)), k.first[0][2], x2);
    cube(x2, k.y2_round0);
    k.partial0 = from_host_mont(h.partial[0]);
    k.kd0 = from_host_mont(h.partial[1]);
    for (int i = 0; i < kLimbs; i++) k.kd0.l[i] += consts::d4(i);
    partial_constants(h);
    felt x{{1, 0, 0, 0}};
    for (int i = 0; i < 522; i++) x = felt_add(x, x);
    r2 = from_canonical(x);
    one = fe{};
    one.l[0] = 1;
  }
};

inline const setup& host_setup() {
  static const setup s;
  return s;
}

}  // namespace f9
}  // namespace gkr
