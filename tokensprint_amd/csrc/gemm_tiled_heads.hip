// The q/k/v projection of a prompt's portion with the q/k preparation in its epilogue
// (gemm_tiled_kernel.h, HEADS): the tiles of 128 columns are a head each.
#include "gemm_tiled_kernel.h"

extern "C" int ts_gemm_tiled_scaled_fits(int M, int N, int K, int pair, int parts);

namespace {

// The estimate of a product's time in one of the two tiles that hold a head, or in any.
float heads_estimate(int M, int N, int K, bool any, int* tile) {
  float best_us = -1.f;
  for (const TileCost& t : kTileCosts) {
    if (!any && t.bn != 128) continue;
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
// of its tile, 2.5 us of epilogue, that of the tile which the product would take, and the preparation
// kernel's time.  One kernel and two, 4,096 columns (24 + 8 heads), K = 1,024, weights from memory, us:
// 300 rows 14.6 / 13.8, 512 15.0 / 15.4, 800 15.9 / 20.8, 1,024 16.7 / 21.7, 1,500 24.9 / 29.3, 2,048
// 26.2 / 32.4, 2,500 40.2 / 40.4 (left separate), 3,000 43.2 / 49.1, 4,096 47.3 / 58.8, 8,192 91.3 / 109.0.
// Rows below 512 are prepared in eager steps only, which wait for the host: a launch less is more than
// the microsecond or two that a tile of half the columns would save (72 rows 13.4 / 11.7).
extern "C" int ts_gemm_tiled_heads_fits(int M, int N, int K, int parts, int hd, int page_size) {
  if (hd != 128 || N % 128 != 0 || page_size <= 0 || !ts_gemm_tiled_scaled_fits(M, N, K, 0, parts)) return 0;
  const float prepare_us = 3.5f + 7.f * ((float)M * N / (2048.f * 4096.f)), host_us = M < 512 ? 4.f : 0.f;
  return heads_estimate(M, N, K, false, nullptr) + 2.5f <=
         heads_estimate(M, N, K, true, nullptr) + prepare_us + host_us;
}

// q, and k and v into their pages, of rows[M, K] W[N, K]^T (ts_gemm_tiled_scaled_bf16's rows and sums),
// W the weights of nq query heads, nkv key heads and nkv value heads of 128, as ts_qk_prepare would make
// them from that product in bfloat16.  `tile`: 0, or 1 or 2 by name (the same to the bit).
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
  if (tile == 0) heads_estimate(M, g.N, K, false, &tile);
  if (tile == 1) return launch_tiled<256, 128, 4, 2, 3, false, bf16_t, kHeads>(g, stream);
  if (tile == 2) return launch_tiled<128, 128, 2, 4, 4, false, bf16_t, kHeads>(g, stream);
  TS_FAIL("gemm_tiled_heads: no tile %d", tile);
}
