// Entry points of the LDS-tiled product for many rows (gemm_tiled_kernel.h): the plain
// form and the gate/up form with the SiLU-multiply in its epilogue.
#include "gemm_tiled_kernel.h"

// 1 if ts_gemm_tiled_bf16 takes these sizes.
extern "C" int ts_gemm_tiled_fits(int M, int N, int K, int pair) {
  const int64_t rows_w = pair ? 2 * (int64_t)N : N;
  return M > 0 && N > 0 && K >= 256 && K % 64 == 0 && N % 16 == 0 &&
         (int64_t)M * K * 2 < (1ll << 32) && rows_w * K * 2 < (1ll << 32);
}

// Per cent of the rounds of the units that the product's elements fill in the tile that its sizes
// take: what edges and a last round leave empty is time in which the library, whose kernels share
// a tile's K out over units, gets ahead.
extern "C" int ts_gemm_tiled_fill(int M, int N, int K, int pair) {
  if (!ts_gemm_tiled_fits(M, N, K, pair)) return 0;
  TiledArgs g{};
  g.M = M, g.N = N, g.K = K;
  const int tile = cheapest_tile(g, pair), units = compute_units();
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
// the library's.  Both timed at 65 to 8,192 rows of 18 weights (N 1,024 to 10,304, K 1,024 to
// 25,600), the weights in memory, bfloat16 out: where N is no multiple of 256 (4,384, 4,640,
// 6,176, 10,304) this kernel takes 0.59 to 1.11 of the library's time, 0.86 in the mean; where
// N is one and the product fills four fifths of its tiles' rounds 0.54 to 1.07, 0.97 in the mean
// (5,120 x 25,600 at 8,192 rows 1,610 / 2,090 us; below four fifths 1.01 in the mean and up to
// 1.30), but for products that the library's tile of 256 x 256 cuts in whole rounds of the units:
// 0.97 to 1.11, 1.08 in the mean, so those stay the library's (with float32 out, whose stores it
// does worse, they do not: 2,048 x 8,192 x 2,048 59 / 66 us).
extern "C" int ts_gemm_tiled_ahead(int M, int N, int K, int c_type) {
  if (!ts_gemm_tiled_fits(M, N, K, 0)) return 0;
  if (N % 256 != 0) return 1;
  const int64_t squares = (int64_t)((M + 255) / 256) * (N / 256);
  if (c_type == TS_BF16 && squares % compute_units() == 0) return 0;
  return ts_gemm_tiled_fill(M, N, K, 0) >= 80;
}

// C[M, N] = A[M, K] W[N, K]^T, or with `pair` C[M, N] = silu(A Wg^T) * (A Wu^T) (or, with a
// `limit` other than 0, gated_unit's other forms) for W = [Wg; Wu] of 2 N rows.  `c_type`: bfloat16 or float32 (float32 not with `pair`).
// `tile`: 0 lets the sizes choose; 1 to 5 name a tile (for measuring; the result is the
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
