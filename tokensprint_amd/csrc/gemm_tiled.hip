// Entry points of the LDS-tiled product for many rows (gemm_tiled_kernel.h): the plain
// form and the gate/up form with the SiLU-multiply in its epilogue.
#include "gemm_tiled_kernel.h"

// 1 if ts_gemm_tiled_bf16 takes these sizes.
extern "C" int ts_gemm_tiled_fits(int M, int N, int K, int pair) {
  const int64_t rows_w = pair ? 2 * (int64_t)N : N;
  return M > 0 && N > 0 && K >= 256 && K % 64 == 0 && N % 16 == 0 &&
         (int64_t)M * K * 2 < (1ll << 32) && rows_w * K * 2 < (1ll << 32);
}

// Per cent of the rounds of the units that the product's elements fill in the tile of 128 rows or more
// that its sizes take: what edges and a last round leave empty is time in which the library, whose kernels share
// a tile's K out over units, gets ahead.
extern "C" int ts_gemm_tiled_fill(int M, int N, int K, int pair) {
  if (!ts_gemm_tiled_fits(M, N, K, pair)) return 0;
  TiledArgs g{};
  g.M = M, g.N = N, g.K = K;
  const int tile = cheapest_tile(g, pair, 128), units = compute_units();
  const int64_t cols = pair ? 2 * (int64_t)N : N;
  for (const TileCost& t : kTileCosts) {
    if (t.tile != tile) continue;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((cols + t.bn - 1) / t.bn);
    const int64_t rounds = (tiles + units - 1) / units;
    return (int)(100 * ((double)M * cols) / ((double)rounds * units * t.bm * t.bn));
  }
  return 0;
}

// 1 if the plain product of these sizes (that ts_gemm_tiled_fits) is this kernel's rather than
// the library's, which shares a tile's K out over units where there are few tiles.  Both timed at
// 65 to 8,192 rows, the weights in memory; times of the library's.
// N no multiple of 256, N 16 to 10,304: the longer K, the more of the tiles' rounds has to be
// filled.  K = 512 0.22 to 1.01 from 48 columns; K = 1,024 0.74 to 0.92 from 1,296 columns, 1.1 to
// 1.3 below with less than a quarter filled; K = 2,048 below 512 rows 0.79 to 1.06 from a half on, 0.92 in
// the mean, and up to 128 rows of at least 6,176 columns 0.93 to 1.00, up to 1.8 else; from 512 rows 0.78 to
// 1.05 from two thirds on, up to 1.13 below;
// K = 4,096 and 8,192 0.81 to 1.01 from seven tenths on (up to 1,024 rows of up to 4,096 columns of
// 4,096 0.90 to 1.04 from a half on), up to 3.4 below (65 rows of 64 columns of 8,192).  151,936
// columns: 0.82 to 0.95 from seven tenths on, up to 1.11 below.
// N a multiple of 256, float32 out: 0.87 to 1.06 from four fifths filled, 0.95 in the mean.  bfloat16
// out, timed at 74 row counts of eight weights (N 2,048 to 10,240, K 2,048 to 25,600): where the
// tiles are 128 x 128 or smaller and four fifths filled 0.62 to 1.00; with larger ones the
// library's 256 x 256 mostly is as good or ahead (0.97 to 1.17), but for long K, where it often
// falls to half of its rate.  K from 5,120: one round of 256 x 128 three quarters filled 0.54 to 1.04,
// and two to three rounds of 256 x 256 0.65 to 1.11, 0.83 in the mean.  K = 12,288 and 25,600: more
// than one such round 0.59 to 1.09, 0.80 in the mean, filled by two thirds (tiles of 256 x 128 in
// several rounds 1.11 to 1.19).  K = 25,600: one round of up to 256 x 128 0.65 to 0.97 whatever it fills
// (5,120 columns, 1,536 rows 338 / 507 us), of larger tiles 0.58 to 1.10, 0.88 in the mean.
// N a multiple of 256 in the small tiles (64 x 64 and 64 x 32), timed at 65 to 1,500 rows of 13 weights (N 512
// to 9,216): K up to 2,048 0.49 to 0.97, 0.70 in the mean, whatever they fill (against the fastest of the
// library's first eight algorithms 0.57 to 0.92 at 65 to 600 rows of five of them); K = 4,096 0.80 to 0.94
// above 256 rows, 1.03 to 1.27 below; K = 8,192 0.90 to 1.38.  Float32 results only up to K = 1,024: above, the
// library shares K out where there are few tiles (at 65 to 513 rows of up to 3,072 columns, by no rule of
// sizes) and is half as far from float64 as one chain of K (K = 2,048 1.3e-7 and 2.7e-7); up to there both
// are one chain (2,362 sizes).
extern "C" int ts_gemm_tiled_ahead(int M, int N, int K, int c_type) {
  if (!ts_gemm_tiled_fits(M, N, K, 0)) return 0;
  TiledArgs g{};
  g.M = M, g.N = N, g.K = K;
  const int small = cheapest_tile(g, false);
  if (N % 256 == 0 && (small == 7 || small == 8) && (c_type == TS_BF16 || K <= 1024))
    return K <= 2048 || (K <= 4096 && M > 256);
  const int tile = cheapest_tile(g, false, 128), units = compute_units();
  const int fill = ts_gemm_tiled_fill(M, N, K, 0);
  if (N % 256 != 0) {
    if (N < 16384 && (K <= 512 ? N >= 48 : K <= 1024 && N >= 1280)) return 1;
    if (N < 16384 && K < 2240) return M <= 128 && N >= 6144 ? 1 : fill >= (M < 512 ? 3 * K / 128 : K / 32);
    return fill >= (K <= 6144 && N <= 4096 && M <= 1024 ? 49 : 70);
  }
  if (c_type != TS_BF16 && fill >= 80) return 1;
  int64_t area = 0, tiles = 0;
  for (const TileCost& t : kTileCosts) {
    if (t.tile != tile) continue;
    area = t.bm * t.bn, tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
  }
  const int64_t squares = (int64_t)((M + 255) / 256) * (N / 256);
  if (K >= 12288 && squares > units) return area != 256 * 128 && fill >= 66;
  if (K >= 5120 && squares > 2 * units && squares <= 3 * units) return fill >= 73;
  if (K >= 16384) return fill >= (area <= 256 * 128 ? 45 : 60);
  if (area == 256 * 128) return K >= 5120 && tiles <= units && fill >= 75;
  return area <= 128 * 128 && fill >= 80;
}

// C[M, N] = A[M, K] W[N, K]^T, or with `pair` C[M, N] = silu(A Wg^T) * (A Wu^T) (or, with a
// `limit` other than 0, gated_unit's other forms) for W = [Wg; Wu] of 2 N rows.  `c_type`: bfloat16 or float32 (float32 not with `pair`).
// `tile`: 0 lets the sizes choose; 1 to 8 name a tile (for measuring; the result is the
// same to the bit).
extern "C" int ts_gemm_tiled_bf16(const void* a, const void* w, void* c, int c_type, int M, int N,
                                  int K, int pair, int tile, float limit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!ts_gemm_tiled_fits(M, N, K, pair))
    TS_FAIL("gemm_tiled: M=%d N=%d K=%d not taken (K a multiple of 64 from 256, N of 16, "
            "operands below 4 GiB)", M, N, K);
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) & 15)
    TS_FAIL("gemm_tiled: operands must be 16-byte aligned");
  TiledArgs g{(const bf16_t*)a, (const bf16_t*)w, c, M, N, K, 0, 0, 1};
  g.limit = limit;
  if (pair) {
    if (c_type != TS_BF16) TS_FAIL("gemm_tiled: the paired form writes bfloat16");
    return choose_tile<true, bf16_t>(g, tile, stream);
  }
  if (c_type == TS_BF16) return choose_tile<false, bf16_t>(g, tile, stream);
  if (c_type == TS_F32) return choose_tile<false, float>(g, tile, stream);
  TS_FAIL("gemm_tiled: output type %d", c_type);
}
