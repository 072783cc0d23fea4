// The q/k/v projection of a prompt's portion with the q/k preparation in its epilogue
// (gemm_tiled_kernel.h, HEADS): the tiles of 128 columns are a head each.
#include "gemm_tiled_kernel.h"

extern "C" int ts_gemm_tiled_scaled_fits(int M, int N, int K, int pair, int parts);

namespace {

// The tiles that hold a head; the smallest for the rows for which the plain forms have 128 x 64, whose
// loads it has.
constexpr TileCost kHeadTiles[] = {
    {6, 64, 128, 1.2f, 0.329f, 0.f}, {2, 128, 128, 2.4f, 0.491f, 0.f}, {1, 256, 128, 4.5f, 0.721f, 0.f}};

// The estimate of a product's time in the best of some tiles.
template <int COUNT>
float estimate(int M, int N, int K, const TileCost (&costs)[COUNT], int* tile) {
  float best_us = -1.f;
  for (const TileCost& t : costs) {
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const int64_t rounds = (tiles + compute_units() - 1) / compute_units();
    const float us = rounds * (t.fixed_us + t.step_us * (K / 64));
    if (best_us < 0.f || us < best_us) {
      best_us = us;
      if (tile) *tile = t.tile;
    }
  }
  return best_us;
}

}  // namespace

// 1 if ts_gemm_tiled_heads_bf16 takes a projection of these sizes and is the faster way: by the estimate
// of its tile, 2.5 us of epilogue (1.7 to 4.2 by the tile), that of the tile which the product would take, and the preparation
// kernel's time.  Rows below 512 are prepared in eager steps only, which wait for the host: four
// microseconds more for a launch less.  One kernel and two, 4,096 columns (24 + 8 heads), K = 1,024, weights from memory, us:
// 72 rows 10.0 / 11.7, 300 10.3 / 13.8, 512 11.0 / 15.5, 800 16.0 / 21.0, 1,024 16.7 / 21.9, 1,500 25.0 /
// 29.4, 2,048 26.6 / 32.4, 2,500 40.6 / 41.4, 4,096 48 / 58, 8,192 92 / 103.  (128 x 128 as the smallest
// tile: 300 rows 14.4.)
extern "C" int ts_gemm_tiled_heads_fits(int M, int N, int K, int parts, int hd, int page_size) {
  if (hd != 128 || N % 128 != 0 || page_size <= 0 || !ts_gemm_tiled_scaled_fits(M, N, K, 0, parts)) return 0;
  const float prepare_us = 3.5f + 7.f * ((float)M * N / (2048.f * 4096.f)), host_us = M < 512 ? 4.f : 0.f;
  return estimate(M, N, K, kHeadTiles, nullptr) + 2.5f <=
         estimate(M, N, K, kTileCosts, nullptr) + prepare_us + host_us;
}

// q, and k and v into their pages, of rows[M, K] W[N, K]^T (ts_gemm_tiled_scaled_bf16's rows and sums),
// W the weights of nq query heads, nkv key heads and nkv value heads of 128, as ts_qk_prepare would make
// them from that product in bfloat16.  `tile`: 0, or 1, 2 or 6 by name (the same to the bit).
extern "C" int ts_gemm_tiled_heads_bf16(const void* rows, const float* sumsq, int parts, float eps,
                                        const void* w, const QkPrepareArgs* heads, int M, int K,
                                        int tile, hipStream_t stream) {
  if (M <= 0) return 0;
  TiledHeadsArgs g{};
  g.heads = *heads;
  const QkPrepareArgs& h = g.heads;
  if (h.nq <= 0 || h.nkv <= 0 || h.num_tokens != M)
    TS_FAIL("gemm_tiled_heads: heads nq=%d nkv=%d, %d tokens of %d", h.nq, h.nkv, h.num_tokens, M);
  const int64_t N = ((int64_t)h.nq + 2 * (int64_t)h.nkv) * h.hd;
  if (h.hd != 128 || N > 1 << 24 || !ts_gemm_tiled_scaled_fits(M, (int)N, K, 0, parts))
    TS_FAIL("gemm_tiled_heads: M=%d K=%d, heads of %d, parts=%d not taken", M, K, h.hd, parts);
  if (!h.q_out || !h.k_dst || !h.v_dst || !h.table || !h.positions || !h.entry_of_token ||
      h.table_width <= 0 || h.page_size <= 0)
    TS_FAIL("gemm_tiled_heads: queries, pages and their table are needed");
  if ((h.cos == nullptr) != (h.sin == nullptr)) TS_FAIL("gemm_tiled_heads: cos and sin go together");
  if (((uintptr_t)rows | (uintptr_t)w | (uintptr_t)h.q_out | (uintptr_t)h.k_dst | (uintptr_t)h.v_dst |
       (uintptr_t)h.cos | (uintptr_t)h.sin) & 15)
    TS_FAIL("gemm_tiled_heads: operands must be 16-byte aligned");
  g.a = (const bf16_t*)rows, g.w = (const bf16_t*)w;
  g.M = M, g.N = (int)N, g.K = K, g.panel = 1;
  g.sumsq_in = sumsq, g.parts = parts, g.eps = eps;
  if (tile == 0) estimate(M, g.N, K, kHeadTiles, &tile);
  if (tile == 1) return launch_tiled<256, 128, 4, 2, 3, false, bf16_t, kHeads>(g, stream);
  if (tile == 2) return launch_tiled<128, 128, 2, 4, 4, false, bf16_t, kHeads>(g, stream);
  if (tile == 6) return launch_tiled<64, 128, 2, 4, 4, false, bf16_t, kHeads>(g, stream);
  TS_FAIL("gemm_tiled_heads: no tile %d", tile);
}
