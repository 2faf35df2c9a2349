// Sumcheck trips over long vectors on the matrix cores.
//
// A trip of three rounds needs the 64 cross sums G[c][c'] = sum_x a_c(x) b_c'(x)
// of its 8 + 8 sub-vectors (k_trip): a contraction over x.  k_trip forms the 64
// QM31 products of an x one by one, about 75 VALU instructions each, which
// outlasts the 256 bytes read, so on long vectors it serves one or two rounds
// per pass over memory.  Here the four words of a value are split into four
// balanced base-256 digits each and the sums of digit products
//   D[(c, word, digit)][(c', word', digit')] = sum_x a-digit * b-digit
// (128 x 128 int32) come from v_mfma_i32_32x32x32_i8: about 30 VALU
// instructions per value whatever the number of rounds, so a pass over memory
// serves three rounds and is bound by HBM.  The digits are combined once per
// workgroup:
//   S[c][c'][word][word'] = sum 256^(digit + digit') D   (mod P),
// and the 16 word products of a pair give its QM31 product.
//
// A workgroup (4 waves) takes 64 x at a time: 1024 values of the 16
// sub-vectors, four per thread (x, x + 16, x + 32, x + 48: lanes read
// consecutive values).  Pending folds are applied as one weighted sum of the
// 2^NP sources (eq weights of the pending challenges as 4 x 4 matrices over
// M31; one partial reduction per source and word instead of a full one per
// product: about 240 instructions for 8 sources against 600 for the seven
// folds).  The digits go to LDS in the MFMA's operand order and each wave
// multiplies one quadrant (4 + 4 sub-vectors).  Two LDS buffers: one barrier
// per 64 x.
//
// LDS order: the operand block of (side, tile of 2 sub-vectors, 32 x) is 1 KB,
// lane l's 16 bytes in slot l: row l % 32 = 16 (c % 2) + 4 word + digit, x
// block l / 32.  A writing instruction has one (word, digit) for all lanes, so
// the slot's low four bits are XORed with the lane's (x block, c % 4): 16
// groups of four lanes then cover the 64 banks once; the reading lanes permute within
// the block.  The K order inside a block is 4 (x % 16) + x / 16, the same on
// both sides.
//
// Measured over 2^28 entries (2 x 4 GiB): the first trip 1348 us (6.4 TB/s, the
// card's plain read rate), the second, which reads them again and writes an
// eighth, 1960 us (4.9 TB/s; its arithmetic alone allows about 4 times that);
// one round per trip took 8 trips of 848 us.  Whole product sumcheck: 2^28
// 6999 -> 3985 us, 2^24 735 -> 508, 2^20 266 -> 244, 2^17 202 -> 192.  Tried,
// against 4.07 ms at that time: cached loads (4.33 ms), four values folded
// together (4.16), three waves per SIMD (spills, 4.50), 256 or 1024 workgroups,
// contiguous or XCD-local ranges per workgroup (no faster).  Eq-sumchecks take the two factors of their
// weight one on each side: the Mul layer of 64 x 13824 (2^20 entries, four
// trips instead of five) 330 -> 309 us, two RMSNorm layers of 64 x 5120 (2^19;
// Part 0 and Part 1) 2204 -> 2164 us.
#pragma once
#include "kernels.h"

namespace gkr {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef int v16i_t __attribute__((ext_vector_type(16)));

constexpr uint64_t kMfmaTripX = 64;           // x per workgroup step
constexpr uint64_t kMfmaTripMaxX = 1u << 16;  // x per workgroup: |digit product sums| <= 2^30

// A value read once by the pass: not kept in the caches.
__device__ __forceinline__ qm31 ld_q_stream(const qm31* p, uint64_t i) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p) + i);
  return qm31{v[0], v[1], v[2], v[3]};
}
// The four balanced digits of a canonical value as signed bytes: centered to
// (-P/2, P/2], so the top digit stays within a byte.
__device__ __forceinline__ uint32_t m31_digits(uint32_t v) {
  const uint32_t top = v >> 30;  // 1: v - P = v + 1 - 2^31
  return (((top << 31) + v) + top + 0x00808080u) ^ 0x00808080u;
}
// 4 x 4 byte transposition: out[d] holds digit d of w[0..3].
__device__ __forceinline__ void transpose4(const uint32_t (&w)[4], uint32_t (&out)[4]) {
  const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
  const uint32_t c = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), d = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
  out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
  out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
  out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
  out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// Multiplication by a constant QM31 e as a matrix over M31 words:
//   y0 = e0 v0 - e1 v1 + f0 v2 - f1 v3     (f0, f1) = (2 + i)(e2, e3)
//   y1 = e1 v0 + e0 v1 + f1 v2 + f0 v3
//   y2 = e2 v0 - e3 v1 + e0 v2 - e1 v3
//   y3 = e3 v0 + e2 v1 + e1 v2 + e0 v3
struct alignas(16) QMat {
  uint32_t e0, e1, e2, e3, f0, f1, ne1, ne3, nf1, pad[3];
};
__device__ __forceinline__ QMat qmat(qm31 e) {
  const cm31 f = cm31_mul_r(qm31_hi(e));
  return QMat{e.a, e.b, e.c, e.d, f.a, f.b, m31_neg(e.b), m31_neg(e.d), m31_neg(f.b), {0, 0, 0}};
}
struct qwide {
  uint64_t y0, y1, y2, y3;
};
// acc += M v; acc below 2^34 a word before, any u64 after (4 (P - 1)^2 + 2^34 < 2^64)
__device__ __forceinline__ void qmat_add(qwide& acc, const QMat& M, qm31 v) {
  acc.y0 += (uint64_t)M.e0 * v.a + (uint64_t)M.ne1 * v.b + (uint64_t)M.f0 * v.c + (uint64_t)M.nf1 * v.d;
  acc.y1 += (uint64_t)M.e1 * v.a + (uint64_t)M.e0 * v.b + (uint64_t)M.f1 * v.c + (uint64_t)M.f0 * v.d;
  acc.y2 += (uint64_t)M.e2 * v.a + (uint64_t)M.ne3 * v.b + (uint64_t)M.e0 * v.c + (uint64_t)M.ne1 * v.d;
  acc.y3 += (uint64_t)M.e3 * v.a + (uint64_t)M.e2 * v.b + (uint64_t)M.e1 * v.c + (uint64_t)M.e0 * v.d;
}
__device__ __forceinline__ uint64_t part_reduce(uint64_t x) { return (x & P) + (x >> 31); }  // below 2^34

// KIND 0 (products) and 1 (eq-weighted products) as k_trip with K = 3; NP
// pending folds (source length n << NP).  Needs n >= 512, a power of two, and
// at most kMfmaTripMaxX x per workgroup.
template <int KIND, int NP>
static __global__ void __launch_bounds__(kBlock, 2) k_trip_mfma(const qm31* __restrict__ sa, const qm31* __restrict__ sb,
                                                         uint64_t n, TripChal al, qm31* __restrict__ da,
                                                         qm31* __restrict__ db, const qm31* __restrict__ eq_hi,
                                                         const qm31* __restrict__ eq_lo, int eq_h, RoundSink sk,
                                                         TripWait tw) {
  if (tw.chal) {  // launched ahead: as k_trip
    const uint32_t st = tw.status[0];
    qm31 ch[kTripMaxK];
#pragma unroll
    for (int r = 0; r < kTripMaxK; r++) ch[r] = ld_q(tw.chal, r);
    __asm__ volatile("" ::: "memory");
    if (st != tw.want) return;
#pragma unroll
    for (int r = 0; r < kTripMaxK; r++)
      if (r < NP) al.c[r] = ch[r];
  }
  __shared__ uint4 buf[2][2][4][2][64];  // [buffer][side][tile][32 x][slot]
  __shared__ QMat wt[1 << NP];
  if constexpr (NP > 0) {
    if (threadIdx.x < (1u << NP)) {  // eq weight of source s: al.c[0] on its top bit
      qm31 e = qm31_one();
#pragma unroll
      for (int l = 0; l < NP; l++)
        e = qm31_mul(e, (threadIdx.x >> (NP - 1 - l)) & 1 ? al.c[l] : qm31_sub(qm31_one(), al.c[l]));
      wt[threadIdx.x] = qmat(e);
    }
    __syncthreads();
  }
  const uint64_t nb = n >> 3;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int side = wave >> 1, c = (wave & 1) * 4 + (lane >> 4), xl = lane & 15;
  const qm31* __restrict__ src = side ? sb : sa;
  qm31* __restrict__ dst = side ? db : da;
  const uint32_t ntile = (uint32_t)(nb / kMfmaTripX);
  // this thread's words in the operand blocks: slot's low bits are (word, digit) ^ swz
  const int swz = ((xl >> 2) * 4 + (c & 3)) & 15;
  const int slot_hi = ((xl >> 2) & 1) * 32 + (c & 1) * 16;
  v16i_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0;
  const int ra = 2 * (wave & 1), rb = 2 * (wave >> 1);  // this wave's quadrant: tiles ra, ra + 1 by rb, rb + 1
  qm31 v[4];
  auto load_plain = [&](uint32_t t) {
    const uint64_t pos = (uint64_t)c * nb + t * kMfmaTripX + xl;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = ld_q_stream(src, pos + 16 * i);
  };
  int p = 0;
  if constexpr (NP == 0) {
    if (blockIdx.x < ntile) load_plain(blockIdx.x);
  }
  for (uint32_t t = blockIdx.x; t < ntile; t += gridDim.x, p ^= 1) {
    const uint64_t x0 = t * kMfmaTripX + xl, pos = (uint64_t)c * nb + x0;
    if constexpr (NP > 0) {
      constexpr int E = 2;  // values folded together: 2 * 2^NP loads in flight
#pragma unroll
      for (int i0 = 0; i0 < 4; i0 += E) {
        qm31 q[1 << NP][E];
#pragma unroll
        for (int s = 0; s < (1 << NP); s++)
#pragma unroll
          for (int i = 0; i < E; i++) q[s][i] = ld_q_stream(src, pos + 16 * (i0 + i) + (uint64_t)s * n);
        qwide f[E];
#pragma unroll
        for (int i = 0; i < E; i++) f[i] = qwide{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < (1 << NP); s++) {
          const QMat M = wt[s];
#pragma unroll
          for (int i = 0; i < E; i++) {
            if (s > 0) {
              f[i].y0 = part_reduce(f[i].y0);
              f[i].y1 = part_reduce(f[i].y1);
              f[i].y2 = part_reduce(f[i].y2);
              f[i].y3 = part_reduce(f[i].y3);
            }
            qmat_add(f[i], M, q[s][i]);
          }
        }
#pragma unroll
        for (int i = 0; i < E; i++)
          v[i0 + i] = qm31{m31_reduce64(f[i].y0), m31_reduce64(f[i].y1), m31_reduce64(f[i].y2), m31_reduce64(f[i].y3)};
      }
      if (dst) {
#pragma unroll
        for (int i = 0; i < 4; i++) st_q(dst, pos + 16 * i, v[i]);
      }
    }
    if constexpr (KIND == 1) {  // eq(x) = hi * lo, one factor on each side
      const uint64_t mask = (1ull << eq_h) - 1;
#pragma unroll
      for (int i = 0; i < 4; i++)
        v[i] = qm31_mul(v[i], side ? ld_q(eq_lo, (x0 + 16 * i) & mask) : ld_q(eq_hi, (x0 + 16 * i) >> eq_h));
    }
    uint32_t* blk = reinterpret_cast<uint32_t*>(buf[p][side][c >> 1][xl >> 3]) + (xl & 3);
#pragma unroll
    for (int w = 0; w < 4; w++) {
      uint32_t d[4], o[4];
#pragma unroll
      for (int i = 0; i < 4; i++) d[i] = m31_digits(w == 0 ? v[i].a : w == 1 ? v[i].b : w == 2 ? v[i].c : v[i].d);
      transpose4(d, o);
#pragma unroll
      for (int k = 0; k < 4; k++) blk[4 * (slot_hi + ((4 * w + k) ^ swz))] = o[k];
    }
    __syncthreads();
    if constexpr (NP == 0) {  // the next values travel while the matrix cores work
      if (t + gridDim.x < ntile) load_plain(t + gridDim.x);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      v4i_t A[2], B[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int hi = lane & 48;  // x block and c % 2
        const int ga = ((ks * 2 + (lane >> 5)) * 4 + ((ra + i) & 1) * 2 + ((lane >> 4) & 1)) & 15;
        const int gb = ((ks * 2 + (lane >> 5)) * 4 + ((rb + i) & 1) * 2 + ((lane >> 4) & 1)) & 15;
        A[i] = *reinterpret_cast<const v4i_t*>(&buf[p][0][ra + i][ks][hi + ((lane & 15) ^ ga)]);
        B[i] = *reinterpret_cast<const v4i_t*>(&buf[p][1][rb + i][ks][hi + ((lane & 15) ^ gb)]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[i], B[j], acc[i][j], 0, 0, 0);
    }
  }
  // Register 4 q + k of lane l holds row 8 q + 4 (l / 32) + k, column l % 32:
  // digit k of (c % 2 = q / 2, word 2 (q % 2) + l / 32) by digit l % 4 of
  // (c' % 2 = (l % 32) / 16, word' (l % 16) / 4).
  __syncthreads();
  uint32_t(*S)[8][16] = reinterpret_cast<uint32_t(*)[8][16]>(buf);  // [c][c'][4 word + word']
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        int64_t s = 0;  // |s| < 2^56
#pragma unroll
        for (int k = 0; k < 4; k++) s += (int64_t)acc[i][j][4 * q + k] << (8 * k);
        uint32_t r = m31_reduce64((uint64_t)(s + ((int64_t)P << 26)));
        r = m31_reduce62((uint64_t)r << (8 * (lane & 3)));
        r = m31_add_xor<1>(r);
        r = m31_add_xor<2>(r);
        if ((lane & 3) == 0)
          S[2 * (ra + i) + q / 2][2 * (rb + j) + ((lane & 31) >> 4)][4 * (2 * (q % 2) + (lane >> 5)) + ((lane & 15) >> 2)] = r;
      }
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint32_t* w = S[threadIdx.x >> 3][threadIdx.x & 7];
    const cm31 t{m31_sub(w[10], w[15]), m31_add(w[11], w[14])};
    const cm31 lo = cm31_add(cm31{m31_sub(w[0], w[5]), m31_add(w[1], w[4])}, cm31_mul_r(t));
    const cm31 hi{m31_add(m31_sub(w[2], w[7]), m31_sub(w[8], w[13])),
                  m31_add(m31_add(w[3], w[6]), m31_add(w[9], w[12]))};
    st_q(sk.partials, (uint64_t)blockIdx.x * 64 + threadIdx.x, qm31_make(lo, hi));
  }
}

}  // namespace gkr
