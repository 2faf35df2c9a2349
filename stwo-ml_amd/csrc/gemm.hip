// Forward-pass M31 matrix product on the matrix cores (the witness).
#include "internal.h"
#include "gemm.h"
/* ------------------------------------------------------------------ forward GEMM
 * C = A * B mod P for canonical M31 matrices (gemm.h).  B's digit planes (only
 * up to its highest non-zero plane) are built once per matrix and kept with
 * it; A's four planes are built per call into a context slot.  One wave per 32 x 32 tile
 * of C (int8-range operands: up to 4 x 2 tiles) and K split; the splits (each at most
 * 16384 deep) are added by k_gemm_reduce. */
static int digit_planes_needed(gkr_ctx* c, const uint32_t* X, uint64_t count, int* nplanes) {
  uint32_t* dmask;
  TRY(ensureT(c, S_GEMMP, 1, &dmask));
  HIP_TRY(hipMemsetAsync(dmask, 0, 4, c->stream));
  const bool vec = ((uintptr_t)X & 15) == 0;
  const dim3 grid((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((count / (vec ? 4 : 1) + 255) / 256, 4096)));
  if (vec)
    GKR_LAUNCH(c, k_digit_mask<true>, grid, dim3(256), 0, X, count, dmask);
  else
    GKR_LAUNCH(c, k_digit_mask<false>, grid, dim3(256), 0, X, count, dmask);
  HIP_TRY(hipGetLastError());
  uint32_t mask = 0;
  HIP_TRY(hipMemcpyAsync(&mask, dmask, 4, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  int np = 1;
  for (int p = 0; p < 4; p++)
    if (mask & (1u << p)) np = p + 1;
  *nplanes = np;
  return GKR_OK;
}

static int pack_planes(gkr_ctx* c, const uint32_t* X, uint64_t outer, uint64_t K, bool kmajor, int np, int8_t* out,
                       uint32_t* mask = nullptr, uint32_t* clear = nullptr) {
  const uint64_t ntiles = (outer + kGemmTile - 1) / kGemmTile, nsteps = (K + kGemmK - 1) / kGemmK;
  const uint64_t slots = ntiles * nsteps * 64;
  const dim3 grid((uint32_t)((slots + 255) / 256));
  if (!kmajor && K % 4 == 0 && ((uintptr_t)X & 15) == 0)
    GKR_LAUNCH(c, k_digit_pack<true>, grid, dim3(256), 0, X, outer, K, kmajor, np, ntiles, nsteps, out, mask, clear);
  else
    GKR_LAUNCH(c, k_digit_pack<false>, grid, dim3(256), 0, X, outer, K, kmajor, np, ntiles, nsteps, out, mask, clear);
  HIP_TRY(hipGetLastError());
  return GKR_OK;
}

static int weight_planes(gkr_ctx* c, gkr_matrix* b) {
  if (b->bplanes) return GKR_OK;
  int np;
  TRY(digit_planes_needed(c, b->dev, b->rows * b->cols, &np));
  const uint64_t ntiles = (b->cols + kGemmTile - 1) / kGemmTile, nsteps = (b->rows + kGemmK - 1) / kGemmK;
  int8_t* d = nullptr;
  HIP_TRY(hipMalloc(&d, (size_t)np * ntiles * nsteps * kGemmBlockBytes));
  const int rc = pack_planes(c, b->dev, b->cols, b->rows, true, np, d);
  if (rc != GKR_OK) {
    drain(c);
    (void)hipFree(d);
    return rc;
  }
  b->bplanes = d;
  b->bnplanes = np;
  return GKR_OK;
}

static int matmul_forward(gkr_ctx* c, const gkr_matrix* a, gkr_matrix* b, uint32_t* C) {
  const uint64_t m = a->rows, k = a->cols, n = b->cols;
  TRY(weight_planes(c, b));
  const uint64_t nsteps = (k + kGemmK - 1) / kGemmK;
  const uint64_t rtiles = (m + kGemmTile - 1) / kGemmTile, ctiles = (n + kGemmTile - 1) / kGemmTile;
  const uint64_t a_plane = rtiles * nsteps * kGemmBlockBytes, b_plane = ctiles * nsteps * kGemmBlockBytes;
  // A: all four planes packed (A is small) with its non-zero mask on the device;
  // B: 1 plane (int8-range weights) or 4
  const int PB = b->bnplanes == 1 ? 1 : 4;
  int8_t* ap;
  TRY(ensureT(c, S_GEMMA, (size_t)4 * a_plane, &ap));
  // two mask words, used in turn: the packing of one product clears the other's
  if (!c->gemm_mask) {
    drain(c);
    uint32_t* w = nullptr;
    HIP_TRY(hipMalloc(&w, 2 * sizeof(uint32_t)));
    if (hipMemsetAsync(w, 0, 2 * sizeof(uint32_t), c->stream) != hipSuccess) {
      (void)hipFree(w);
      return fail(GKR_ERR_DEVICE, "clear of the digit masks failed");
    }
    c->gemm_mask = w;
  }
  uint32_t* amask = c->gemm_mask + (c->gemm_turn & 1);
  uint32_t* next_mask = c->gemm_mask + (~c->gemm_turn & 1);
  c->gemm_turn++;
  TRY(pack_planes(c, a->dev, m, k, false, 4, ap, amask, next_mask));
  const int8_t* bp = b->bplanes;
  if (PB > b->bnplanes) {  // a 2- or 3-plane weight: extend with zero planes in scratch
    int8_t* ext;
    TRY(ensureT(c, S_GEMMB, (size_t)4 * b_plane, &ext));
    HIP_TRY(hipMemcpyAsync(ext, b->bplanes, (size_t)b->bnplanes * b_plane, hipMemcpyDeviceToDevice, c->stream));
    HIP_TRY(hipMemsetAsync(ext + (size_t)b->bnplanes * b_plane, 0, (size_t)(4 - b->bnplanes) * b_plane, c->stream));
    bp = ext;
  }
  const uint64_t waves = rtiles * ctiles, blocks_x = (waves + 3) / 4;
  // Int8-range operands: the wave's tiles by the work there is, counted in steps
  // of one 32 x 32 tile of C by 32 of K.  A call of few steps is bound by latency
  // and launches: one tile per wave, which needs no k_gemm_a4 behind it (us per
  // call with one tile and with the wider ones: 512 x 576 x 1536 23.7, 29.0; 512 x
  // 64 x 64 21.3, 24.4; 256 x 2560 x 5120 32.6, 42.3; 64 x 5120 x 1024 24.2, 28.8).
  // Above, wider tiles read fewer operands (one tile per wave in 2048 workgroups by
  // K splits before -> now, weights of 5120 x 13824): 4 x 2 from 8 row tiles (m =
  // 512: 232.5 -> 67.4), 2 x 2 from 4 (m = 128: 83.9 -> 43.2), 2 x 1 from 2 (m =
  // 64: 63.5 -> 42.1), 1 x 1 for one (m = 1: 41.2 -> 29.7).  The lines, by one tile
  // and wider for A of one plane and of four: from 4 row tiles 2^18 steps (256 x
  // 5120 x 5120, 204,800 steps: 40.4, 44.8 and 103, 86; 512 x 5120 x 13824,
  // 1,105,920: 96.8, 66.5 and 302, 258), below 2^16 (64 x 5120 x 5120, 51,200: 27.8,
  // 32.1 and 45.4, 46.5; 64 x 5120 x 13824, 138,240: 32.6, 41.6 and 65.9, 60.4).
  // K is split only where the tiles alone give under 576 waves, and then into
  // about 768 waves (512 and 1024 up to 1.3 times slower for one shape or another):
  // a split writes and reads its partial sums.  With one tile per wave
  // of more than 80 steps, up to 5 splits (or of 40 steps) are made for 1536 waves:
  // a wave's chain of steps is what an A of four planes waits for (in 2048
  // workgroups, by the rule for 768 waves, now: 1 x 5120 x 13824 49.4, 59.3, 43.2;
  // 128 x 5120 x 5120 75.8, 70.2, 56.8; 1 x 3000 x 11000 34.2, 39.6, 31.0), and an A
  // of one plane loses little (1 x 13824 x 5120 30.8 -> 31.5).  For the same reason
  // chains over 256 steps are halved where the tiles are under 2048 (96 x 13824 x
  // 13824: 206, 236, 206; A of one plane 129, 108, 76).
  const bool wide = waves * nsteps >= (rtiles >= 4 ? 1ull << 18 : 1ull << 16);
  const int RT = !wide ? 1 : rtiles >= 8 ? 4 : rtiles >= 2 ? 2 : 1, CT = wide && rtiles >= 4 ? 2 : 1;
  const int WR = wide && rtiles >= 4 ? 2 : 1;
  const uint64_t rgroups = (rtiles + RT * WR - 1) / (RT * WR), cgroups = (ctiles + CT * (4 / WR) - 1) / (CT * (4 / WR));
  const uint64_t tile_waves = (rtiles + RT - 1) / RT * ((ctiles + CT - 1) / CT);
  uint64_t splits = PB == 1 ? (tile_waves >= 576 ? 1 : (768 + tile_waves - 1) / tile_waves)
                            : (2048 + blocks_x - 1) / blocks_x;
  if (PB == 1 && nsteps > 256 * splits && waves * splits < 2048) splits *= 2;
  if (PB == 1 && RT * CT == 1 && nsteps > 80 && tile_waves < 1024)
    splits = std::max(splits, std::min<uint64_t>(std::max<uint64_t>(5, nsteps / 40), (1536 + tile_waves - 1) / tile_waves));
  splits = std::min<uint64_t>(splits, std::max<uint64_t>(1, nsteps / 16));
  splits = std::max<uint64_t>(splits, (nsteps * kGemmK + kGemmMaxKPass - 1) / kGemmMaxKPass);
  const uint64_t sps = (nsteps + splits - 1) / splits;
  splits = (nsteps + sps - 1) / sps;
  if (blocks_x > 0x7fffffffull || nsteps > 0xffffffffull || splits > 65535)
    return fail(GKR_ERR_INVALID, "forward GEMM: grid too large");
  uint32_t* part = C;
  if (splits > 1) TRY(ensureT(c, S_GEMMP, splits * m * n, &part));
  if (PB == 1) {
    auto int8_launch = [&](auto kernel) {
      uint32_t rg;
      const dim3 grid = gemm_group_grid(rgroups, cgroups, splits, &rg);
      GKR_LAUNCH(c, kernel, grid, dim3(256), 0, ap, a_plane, amask, bp, m, n, (uint32_t)nsteps, (uint32_t)rtiles,
                 (uint32_t)ctiles, rg, (uint32_t)cgroups, (uint32_t)sps, part);
    };
    if (RT == 4)
      int8_launch(k_gemm_int8<4, 2, 2>);
    else if (CT == 2)
      int8_launch(k_gemm_int8<2, 2, 2>);
    else if (RT == 2)
      int8_launch(k_gemm_int8<2, 1, 1>);
    else
      int8_launch(k_gemm_int8<1, 1, 1>);
    auto a4_launch = [&](auto kernel, uint64_t ct) {
      uint32_t rg;
      const uint64_t groups = (ctiles + 4 * ct - 1) / (4 * ct);
      const dim3 grid = gemm_group_grid(rtiles, groups, splits, &rg);
      GKR_LAUNCH(c, kernel, grid, dim3(256), 0, ap, a_plane, amask, bp, m, n, nsteps, (uint32_t)rtiles, (uint32_t)ctiles,
                 rg, (uint32_t)groups, sps, part);
    };
    // two column tiles per wave in chains of 80 steps and with columns for every
    // wave (one, two, us: 64 x 5120 x 13824 67.5, 60.4; 200 x 13824 x 5120 168, 142;
    // 512 x 8192 x 8192 305, 242; 384 x 3000 x 11000, 47 steps, 133, 147; 16384 x 5120 x
    // 128, 4 column tiles, 287, 360)
    if (RT * CT > 1 && ctiles >= 32 && sps >= 80)
      a4_launch(k_gemm_a4<2>, 2);
    else if (RT * CT > 1)
      a4_launch(k_gemm_a4<1>, 1);
  } else {
    GKR_LAUNCH(c, k_gemm_m31, dim3((uint32_t)blocks_x, (uint32_t)splits), dim3(256), 0, ap, a_plane, amask, bp, b_plane,
               m, n, nsteps, rtiles, ctiles, sps, part);
  }
  HIP_TRY(hipGetLastError());
  if (splits > 1) {
    const uint64_t count = m * n;
    GKR_LAUNCH(c, k_gemm_reduce, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, part, count, (int)splits, C);
    HIP_TRY(hipGetLastError());
  }
  return GKR_OK;
}

extern "C" int gkr_matmul_forward_into(gkr_ctx* c, const gkr_matrix* a, const gkr_matrix* b, gkr_matrix* out) {
  if (!c || !a || !b || !out || !out->dev) return fail(GKR_ERR_INVALID, "null argument");
  if (a->cols != b->rows || out->rows != a->rows || out->cols != b->cols)
    return fail(GKR_ERR_INVALID, "forward GEMM: A %llux%llu . B %llux%llu into %llux%llu", (unsigned long long)a->rows,
                (unsigned long long)a->cols, (unsigned long long)b->rows, (unsigned long long)b->cols,
                (unsigned long long)out->rows, (unsigned long long)out->cols);
  if (out == a || out == b) return fail(GKR_ERR_INVALID, "forward GEMM: output aliases an input");
  HIP_TRY(hipSetDevice(c->device));
  TRY(drop_derived(c, out));  // the contents change
  return matmul_forward(c, a, const_cast<gkr_matrix*>(b), out->dev);
}

extern "C" int gkr_matmul_forward(gkr_ctx* c, const gkr_matrix* a, const gkr_matrix* b, gkr_matrix** out) {
  if (!c || !a || !b || !out) return fail(GKR_ERR_INVALID, "null argument");
  if (a->cols != b->rows)
    return fail(GKR_ERR_INVALID, "forward GEMM: A is %llux%llu, B is %llux%llu", (unsigned long long)a->rows,
                (unsigned long long)a->cols, (unsigned long long)b->rows, (unsigned long long)b->cols);
  if (a->rows == 0 || a->cols == 0 || b->cols == 0) return fail(GKR_ERR_INVALID, "forward GEMM: empty matrix");
  HIP_TRY(hipSetDevice(c->device));
  uint32_t* d = nullptr;
  HIP_TRY(hipMalloc(&d, a->rows * b->cols * sizeof(uint32_t)));
  int rc = matmul_forward(c, a, const_cast<gkr_matrix*>(b), d);
  if (rc == GKR_OK) rc = sync(c);
  if (rc != GKR_OK) {
    drain(c);
    (void)hipFree(d);
    return rc;
  }
  *out = new_matrix(c, d, a->rows, b->cols, true);
  return GKR_OK;
}

