// Forward-pass M31 matrix product C = A * B mod P on the matrix cores
// (the witness GEMM before the GKR walk; reference: m31_gemm_kernel /
// m31_gemv_kernel, engine/src/gpu_sumcheck.rs:418-460, gpu_matmul_m31_full
// :3104).  Exact for any canonical M31 inputs.
//
// Digit planes.  A value x in [0, P) is centered to v in (-P/2, P/2] and
// written as four balanced signed digits, v = sum_p d_p 256^p, d_p in
// [-128, 127].  Then
//   (A B)_ij = sum_s 256^s sum_{p+q=s} sum_k a_p[i][k] b_q[k][j]   (mod P),
// each inner sum an int8 GEMM on the matrix cores.  A group s holds at most 4
// pairs of products of magnitude <= 2^14, so K <= 16384 per pass stays inside
// int32.  Finally C_ij = sum_s 2^(8s mod 31) * group_s mod P (2^31 = 1 mod P).
// Planes that are zero everywhere are neither stored nor multiplied: int8-range
// data (|v| <= 127: the configs' weights and activations) has plane 0 only,
// so a weight streams 1 byte per entry and a K step costs one MFMA.
//
// Operand blocks.  v_mfma_i32_32x32x32_i8 takes, in lane l, row (A) or column
// (B) l % 32 and the 16 K values 16 (l / 32) .. + 15 of a 32-wide K step (any
// K order shared by A and B gives the same sum).  A plane is stored as 1 KB
// blocks, one per (32-row or 32-column tile, 32-wide K step), with lane l's
// 16 bytes at offset 16 l: one coalesced 16-byte load per lane.  Block (t, c)
// of a plane is at ((t * nsteps) + c) * 1024.  The accumulator holds rows
// 8 (v / 4) + 4 (l / 32) + v % 4 of column l % 32 in register v.
#pragma once
#include <stdint.h>

#include <type_traits>

#include "field.h"

namespace gkr {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kGemmK = 32;     // K per MFMA step
constexpr int kGemmTile = 32;  // rows / columns per wave tile
constexpr int kGemmBlockBytes = 1024;
constexpr uint64_t kGemmMaxKPass = 16384;  // K per accumulation pass (int32 bound)

__device__ __forceinline__ int32_t center_m31(uint32_t x) {
  return x > (P >> 1) ? (int32_t)x - (int32_t)P : (int32_t)x;
}
// Balanced digit p of v (p = 0..3); digits above 0 vanish for |v| <= 127.
__device__ __forceinline__ void balanced_digits(int32_t v, int32_t (&d)[4]) {
#pragma unroll
  for (int p = 0; p < 4; p++) {
    d[p] = (int32_t)(int8_t)(v & 0xff);
    v = (v - d[p]) >> 8;  // exact; after three digits |v| <= 64
  }
}

// Which planes of X (count canonical M31 values, 16-byte aligned when VEC) are
// non-zero: bit p of *mask (zero before the launch).  Grid-stride, an OR
// across the workgroup in LDS, then at most one vector atomic per workgroup.
// 70.8 M values: 505 us with 4-byte loads by 256 workgroups, 71 us with
// 16-byte loads by up to 4096.
template <bool VEC>
static __global__ void __launch_bounds__(256) k_digit_mask(const uint32_t* __restrict__ X, uint64_t count,
                                                    uint32_t* __restrict__ mask) {
  __shared__ uint32_t wave_bits[4];
  uint32_t bits = 0;
  const uint64_t t0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, nt = (uint64_t)gridDim.x * blockDim.x;
  auto take = [&](uint32_t x) {
    int32_t d[4];
    balanced_digits(center_m31(x), d);
#pragma unroll
    for (int p = 0; p < 4; p++) bits |= (d[p] != 0 ? 1u : 0u) << p;
  };
  uint64_t rest = 0;
  if constexpr (VEC) {
    rest = count / 4;
    for (uint64_t i = t0; i < rest; i += nt) {
      const uint4 q = reinterpret_cast<const uint4*>(X)[i];
      take(q.x);
      take(q.y);
      take(q.z);
      take(q.w);
    }
    rest *= 4;
  }
  for (uint64_t i = rest + t0; i < count; i += nt) take(X[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) bits |= __shfl_xor(bits, off);
  if ((threadIdx.x & 63) == 0) wave_bits[threadIdx.x >> 6] = bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t all = wave_bits[0] | wave_bits[1] | wave_bits[2] | wave_bits[3];
    if (all & ~*(volatile const uint32_t*)mask) atomicOr(mask, all);
  }
}

// Pack planes 0..nplanes-1 of X into operand blocks.  kmajor = false: X is
// outer x K row-major (A: outer = row); kmajor = true: X is K x outer
// row-major (B: outer = column).  One thread fills one lane slot (16 bytes
// per plane) of one block; K and outer beyond the matrix are zero.  When mask
// is given (zero before the launch), bit p of 1..3 is set if plane p is non-zero, and
// *clear, the mask word of the next product on the stream, is zeroed.  VEC
// (row-major X, K a multiple of 4, X 16-byte aligned): a slot's 16 values are
// four 16-byte loads (a whole 512 x 5120 x 1024 product 34.0 -> 30.3 us).
template <bool VEC>
static __global__ void __launch_bounds__(256) k_digit_pack(const uint32_t* __restrict__ X, uint64_t outer, uint64_t K,
                                                    bool kmajor, int nplanes, uint64_t ntiles, uint64_t nsteps,
                                                    int8_t* __restrict__ planes, uint32_t* __restrict__ mask,
                                                    uint32_t* __restrict__ clear) {
  __shared__ uint32_t wave_bits[4];
  const uint64_t slot = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;  // (tile, step, lane)
  uint32_t bits = 0;
  if (clear && slot == 0) *clear = 0;
  if (slot < ntiles * nsteps * 64) {
    const int lane = (int)(slot & 63);
    const uint64_t blk = slot >> 6, tile = blk / nsteps, step = blk - tile * nsteps;
    const uint64_t o = tile * kGemmTile + (lane & 31);
    const uint64_t k0 = step * kGemmK + 16 * (lane >> 5);
    uint32_t w[4][4];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
      for (int g = 0; g < 4; g++) w[p][g] = 0;
    uint32_t xs[16];
    if constexpr (VEC) {
      uint4 q[4];
#pragma unroll
      for (int g = 0; g < 4; g++)
        q[g] = o < outer && k0 + 4 * g < K ? *(const uint4*)(X + o * K + k0 + 4 * g) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        xs[4 * g] = q[g].x;
        xs[4 * g + 1] = q[g].y;
        xs[4 * g + 2] = q[g].z;
        xs[4 * g + 3] = q[g].w;
      }
    } else {
#pragma unroll
      for (int t = 0; t < 16; t++) {
        const uint64_t kk = k0 + t;
        xs[t] = o < outer && kk < K ? (kmajor ? X[kk * outer + o] : X[o * K + kk]) : 0u;
      }
    }
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const uint32_t x = xs[t];
      int32_t d[4];
      balanced_digits(center_m31(x), d);
#pragma unroll
      for (int p = 0; p < 4; p++) w[p][t >> 2] |= ((uint32_t)d[p] & 0xffu) << (8 * (t & 3));
    }
    const uint64_t plane_bytes = ntiles * nsteps * kGemmBlockBytes;
    for (int p = 0; p < nplanes; p++) {
      uint4 v;
      v.x = w[p][0];
      v.y = w[p][1];
      v.z = w[p][2];
      v.w = w[p][3];
      *(uint4*)(planes + p * plane_bytes + blk * kGemmBlockBytes + 16 * lane) = v;
    }
#pragma unroll
    for (int p = 0; p < 4; p++) bits |= ((w[p][0] | w[p][1] | w[p][2] | w[p][3]) != 0 ? 1u : 0u) << p;
  }
  if (!mask) return;  // uniform: a kernel argument
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) bits |= __shfl_xor(bits, off);
  if ((threadIdx.x & 63) == 0) wave_bits[threadIdx.x >> 6] = bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    // atomics on one address take about 20 ns each, one after another: only the
    // planes that decide, and only while their bits are missing
    const uint32_t all = (wave_bits[0] | wave_bits[1] | wave_bits[2] | wave_bits[3]) & 0xeu;
    if (all & ~*(volatile const uint32_t*)mask) atomicOr(mask, all);
  }
}

// An int32 digit-product sum (below 2^31 - 1 in magnitude) mod P.
__device__ __forceinline__ uint32_t gemm_mod_p(int32_t x) { return x < 0 ? (uint32_t)(x + (int32_t)P) : (uint32_t)x; }

// One wave: CT 32 x 32 tiles of C, (rt, ct) and the next columns, over K steps
// [s0, s1) from PA / PB planes of A / B (the planes above are zero), U K
// steps' loads issued together.  Canonical sums go to out[row][col].
template <int PA, int PB, int CT, int U>
__device__ __forceinline__ void gemm_tile(const int8_t* __restrict__ Ap, uint64_t a_plane_bytes,
                                          const int8_t* __restrict__ Bp, uint64_t b_plane_bytes, uint64_t m, uint64_t n,
                                          uint64_t nsteps, uint64_t rt, uint64_t ct, uint64_t ctiles, uint64_t s0,
                                          uint64_t s1, uint32_t* __restrict__ out) {
  constexpr int NG = PA + PB - 1;
  const int lane = threadIdx.x & 63;
  v16i acc[CT][NG];
#pragma unroll
  for (int j = 0; j < CT; j++)
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[j][g][v] = 0;
  const int8_t* abase = Ap + (rt * nsteps) * kGemmBlockBytes + 16 * lane;
  const int8_t* bbase[CT];
#pragma unroll
  for (int j = 0; j < CT; j++)  // a tile past the edge reads the last one and is not stored
    bbase[j] = Bp + ((ct + j < ctiles ? ct + j : ctiles - 1) * nsteps) * kGemmBlockBytes + 16 * lane;
  auto step = [&](auto nu, uint64_t s) {
    constexpr int N = decltype(nu)::value;
    v4i a[N][PA], b[N][CT][PB];
#pragma unroll
    for (int u = 0; u < N; u++) {
#pragma unroll
      for (int p = 0; p < PA; p++) a[u][p] = *(const v4i*)(abase + p * a_plane_bytes + (s + u) * kGemmBlockBytes);
#pragma unroll
      for (int j = 0; j < CT; j++)
#pragma unroll
        for (int q = 0; q < PB; q++)
          b[u][j][q] = __builtin_nontemporal_load((const v4i*)(bbase[j] + q * b_plane_bytes + (s + u) * kGemmBlockBytes));
    }
    // Left to itself the compiler waits for the first loads before it issues the
    // rest (one plane of A by four of B, 1 x 5120 x 13824 82.1 -> 66.4 us; four by
    // one, 512 x 5120 x 13824 298 -> 259).  Two steps of four by four planes are
    // long enough to hide it (128 x 5120 x 13824 225 us so, 238 with the barrier).
    if constexpr (PA * PB < 16) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < N; u++)
#pragma unroll
      for (int j = 0; j < CT; j++)
#pragma unroll
        for (int p = 0; p < PA; p++)
#pragma unroll
          for (int q = 0; q < PB; q++)
            acc[j][p + q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][p], b[u][j][q], acc[j][p + q], 0, 0, 0);
  };
  uint64_t s = s0;
  for (; s + U <= s1; s += U) step(std::integral_constant<int, U>{}, s);
  for (; s < s1; s++) step(std::integral_constant<int, 1>{}, s);
#pragma unroll
  for (int j = 0; j < CT; j++) {
    const uint64_t col = (ct + j) * kGemmTile + (lane & 31);
    if (ct + j >= ctiles || col >= n) continue;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const uint64_t row = rt * kGemmTile + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
      if (row >= m) continue;
      uint64_t total = 0;
#pragma unroll
      for (int g = 0; g < NG; g++)
        total += (uint64_t)m31_reduce64((uint64_t)gemm_mod_p(acc[j][g][v]) << ((8 * g) % 31));
      out[row * n + col] = m31_reduce64(total);
    }
  }
}

// The row and column group of a workgroup in a grid of gemm_group_grid:
// workgroups of one XCD (blockIdx 8 apart) take a run of the groups,
// counted down the columns, an eighth of them each, so that those that share
// column tiles share an L2, which then reads B once, and every XCD has as much
// to do (column groups to XCDs in turn: 4096 x 5120 x 64 ran on one of the
// eight, 103.4 us; 50.9 now with one tile per wave).  blockIdx.z counts runs of
// rgroups row groups, for grids that a launch would not take in one dimension.
// False: no group.
__device__ __forceinline__ bool gemm_group(uint32_t rgroups, uint32_t cgroups, uint32_t& rg, uint32_t& cg) {
  const uint64_t at = (uint64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  rg = (uint32_t)(at % rgroups) + blockIdx.z * rgroups;
  cg = (uint32_t)(at / rgroups);
  return cg < cgroups;
}
constexpr uint64_t kGemmMaxGroups = 1ull << 23;  // of 256 threads: half of the 2^32 that a dimension takes
inline dim3 gemm_group_grid(uint64_t rgroups, uint64_t cgroups, uint64_t splits, uint32_t* rgroups_arg) {
  const uint64_t z = rgroups * cgroups / kGemmMaxGroups + 1, rows = (rgroups + z - 1) / z;
  *rgroups_arg = (uint32_t)rows;
  return dim3((uint32_t)((rows * cgroups + 7) / 8 * 8), (uint32_t)splits, (uint32_t)z);
}

// Int8-range operands (one plane each): a workgroup's 4 waves, WR down and
// 4 / WR across, each own RT x CT tiles of C, so a K step's RT + CT operand
// blocks feed RT * CT MFMAs.  One 32 x 32 tile per wave reads 2 KB per MFMA
// (32 cycles of a SIMD), 256 bytes a cycle and CU against the 64 the vector
// cache delivers; 4 x 2 tiles read 0.75 KB.  The next step's blocks are loaded
// while this step's are multiplied; every tile shape sums the same integers.
// Workgroups go to XCDs by gemm_group.
// An A with higher planes (*amask) is for gemm_tile: here where a wave has one
// tile, else in k_gemm_a4, launched behind (one of the two returns at once).
template <int RT, int CT, int WR>
static __global__ void __launch_bounds__(256) k_gemm_int8(const int8_t* __restrict__ Ap, uint64_t a_plane_bytes,
                                                   const uint32_t* __restrict__ amask,
                                                   const int8_t* __restrict__ Bp, uint64_t m, uint64_t n,
                                                   uint32_t nsteps, uint32_t rtiles, uint32_t ctiles, uint32_t rgroups,
                                                   uint32_t cgroups, uint32_t steps_per_split,
                                                   uint32_t* __restrict__ out) {
  constexpr int WC = 4 / WR;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t rg, cg;
  if (!gemm_group(rgroups, cgroups, rg, cg)) return;
  const uint32_t rt0 = (rg * WR + wave % WR) * RT, ct0 = (cg * WC + wave / WR) * CT;
  if (rt0 >= rtiles || ct0 >= ctiles) return;
  const uint32_t split = blockIdx.y, s0 = split * steps_per_split;
  const uint32_t s1 = s0 + steps_per_split < nsteps ? s0 + steps_per_split : nsteps;
  out += (uint64_t)split * m * n;
  if (*amask & 0xeu) {  // uniform
    if constexpr (RT * CT == 1) gemm_tile<4, 1, 1, 4>(Ap, a_plane_bytes, Bp, 0, m, n, nsteps, rt0, ct0, ctiles, s0, s1, out);
    return;
  }
  const int8_t* ab[RT];
  const int8_t* bb[CT];
#pragma unroll
  for (int i = 0; i < RT; i++)  // tiles past the edge read the last one and are not stored
    ab[i] = Ap + (uint64_t)(rt0 + i < rtiles ? rt0 + i : rtiles - 1) * nsteps * kGemmBlockBytes + 16 * lane;
#pragma unroll
  for (int j = 0; j < CT; j++)
    bb[j] = Bp + (uint64_t)(ct0 + j < ctiles ? ct0 + j : ctiles - 1) * nsteps * kGemmBlockBytes + 16 * lane;
  v16i acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0;
  constexpr int U = RT * CT >= 8 ? 6 : 8;  // K steps in flight
  v4i a[U][RT], b[U][CT];
  auto load = [&](int u, uint32_t s) {
    const uint64_t off = (uint64_t)(s < s1 ? s : s1 - 1) * kGemmBlockBytes;  // past the end: read again, unused
#pragma unroll
    for (int i = 0; i < RT; i++) a[u][i] = *(const v4i*)(ab[i] + off);
#pragma unroll
    for (int j = 0; j < CT; j++) b[u][j] = *(const v4i*)(bb[j] + off);
  };
#pragma unroll
  for (int u = 0; u < U; u++) load(u, s0 + u);
  for (uint32_t s = s0; s < s1; s += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (s + u < s1) {  // uniform
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
          for (int j = 0; j < CT; j++)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
        load(u, s + u + U);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < CT; j++) {
      const uint64_t col = (uint64_t)(ct0 + j) * kGemmTile + (lane & 31);
      if (rt0 + i >= rtiles || ct0 + j >= ctiles || col >= n) continue;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const uint64_t row = (uint64_t)(rt0 + i) * kGemmTile + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
        if (row < m) out[row * n + col] = gemm_mod_p(acc[i][j][v]);
      }
    }
}

// A of four planes by a one-plane B: one wave per 32 rows x CT * 32 columns of
// C and K split.  A workgroup's four waves take the same rows, whose four KB a
// K step they then share in the vector cache, and columns next to each other
// (four row tiles of one column instead, both before the barrier in
// gemm_tile: 200 x 13824 x 5120 216 us against 190, 300 x 5120 x 13824 254
// against 227, 512 x 5120 x 13824 320 against 297).
template <int CT>
static __global__ void __launch_bounds__(256) k_gemm_a4(const int8_t* __restrict__ Ap, uint64_t a_plane_bytes,
                                                 const uint32_t* __restrict__ amask, const int8_t* __restrict__ Bp,
                                                 uint64_t m, uint64_t n, uint64_t nsteps, uint32_t rtiles,
                                                 uint32_t ctiles, uint32_t rgroups, uint32_t cgroups,
                                                 uint64_t steps_per_split, uint32_t* __restrict__ out) {
  if (!(*amask & 0xeu)) return;  // uniform
  uint32_t rt, cg;
  if (!gemm_group(rgroups, cgroups, rt, cg)) return;
  const uint32_t ct = (cg * 4 + (threadIdx.x >> 6)) * CT;
  if (rt >= rtiles || ct >= ctiles) return;
  const uint64_t s0 = blockIdx.y * steps_per_split;
  const uint64_t s1 = s0 + steps_per_split < nsteps ? s0 + steps_per_split : nsteps;
  gemm_tile<4, 1, CT, 4>(Ap, a_plane_bytes, Bp, 0, m, n, nsteps, rt, ct, ctiles, s0, s1,
                         out + (uint64_t)blockIdx.y * m * n);
}

// General values: one wave per 32 x 32 tile of C and K split, four planes of
// B.  A's plane count (1 or 4) is read from *amask (its non-zero planes,
// written by the A packing), so no host round trip decides.  Partial sums go
// to out[split][row][col].
static __global__ void __launch_bounds__(256) k_gemm_m31(const int8_t* __restrict__ Ap, uint64_t a_plane_bytes,
                                                  const uint32_t* __restrict__ amask,
                                                  const int8_t* __restrict__ Bp, uint64_t b_plane_bytes,
                                                  uint64_t m, uint64_t n, uint64_t nsteps, uint64_t rtiles,
                                                  uint64_t ctiles, uint64_t steps_per_split,
                                                  uint32_t* __restrict__ out) {
  const uint64_t wave = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wave >= rtiles * ctiles) return;
  const uint64_t rt = wave % rtiles, ct = wave / rtiles;  // the row tiles of a column tile are neighbours
  const uint64_t s0 = blockIdx.y * steps_per_split;
  const uint64_t s1 = s0 + steps_per_split < nsteps ? s0 + steps_per_split : nsteps;
  out += (uint64_t)blockIdx.y * m * n;
  if (*amask & 0xeu)  // uniform
    gemm_tile<4, 4, 1, 2>(Ap, a_plane_bytes, Bp, b_plane_bytes, m, n, nsteps, rt, ct, ctiles, s0, s1, out);
  else
    gemm_tile<1, 4, 1, 4>(Ap, a_plane_bytes, Bp, b_plane_bytes, m, n, nsteps, rt, ct, ctiles, s0, s1, out);
}

// C = sum over splits of the partials, mod P.
static __global__ void k_gemm_reduce(const uint32_t* __restrict__ part, uint64_t count, int splits, uint32_t* __restrict__ C) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint64_t s = 0;
  for (int t = 0; t < splits; t++) s += part[(uint64_t)t * count + i];
  C[i] = m31_reduce64(s);
}

}  // namespace gkr
