// Test-only host build of the limb-level operations of stwo-ml_amd/csrc/felt9.h
// and poseidon9.h on limbs given by the caller (nine u32 each).
#include "../../stwo-ml_amd/csrc/poseidon9_host.h"

using namespace gkr;

namespace {
f9::fe load(const uint32_t* p) {
  f9::fe r;
  for (int k = 0; k < 9; k++) r.l[k] = p[k];
  return r;
}
void store(const f9::fe& a, uint32_t* p) {
  for (int k = 0; k < 9; k++) p[k] = a.l[k];
}
}  // namespace

extern "C" {
void f9_mul_limbs(const uint32_t* a, const uint32_t* b, uint32_t* out) {
  f9::fe r;
  f9::mul(load(a), load(b), r);
  store(r, out);
}
void f9_sqr_limbs(const uint32_t* a, uint32_t* out) {
  f9::fe r;
  f9::sqr(load(a), r);
  store(r, out);
}
// signed limbs on either side
void f9_mul_signed(const uint32_t* a, const uint32_t* b, uint32_t* out) {
  f9::fe r;
  f9::mul<true>(load(a), load(b), r);
  store(r, out);
}
void f9_sqr_signed(const uint32_t* a, uint32_t* out) {
  f9::fe d, r;
  f9::twice(load(a), d);
  f9::sqr2<true>(load(a), d, r);
  store(r, out);
}
// (u, v, x) -> (u', u, x') with the constants of round r
void f9_partial_round(uint32_t* u, uint32_t* v, uint32_t* x, int r) {
  f9::fe U = load(u), V = load(v), X = load(x);
  f9::partial_round(U, V, X, f9::host_setup().k.ku[r], f9::host_setup().k.x6[r]);
  store(U, v);
  store(V, u);
  store(X, x);
}
void f9_ku(int r, uint32_t* out) {
  store(f9::host_setup().k.ku[r], out);
  out[9] = f9::host_setup().k.x6[r];
}
}
