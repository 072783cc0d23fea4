// The convolved form of the product of gemm_direct.hip: C = A W^T in float32, and a range of its
// columns through a short causal convolution with SiLU as they leave, for steps in which every
// row is its entry's only token.  A channel is one column, and its last inputs are read and
// written by the lane that holds its row's result, so nothing crosses between workgroups; the
// convolution as a kernel of its own took 3.9 to 4.8 us behind each product, a launch and three
// dependent trips to memory for a hundred kilobytes; here it adds 0.7 to 1.3 us (8 rows: 10,304 x
// 2,048 weights 12.4 -> 13.7 us, 6,176 x 2,048 9.0 -> 9.7, 2,192 x 2,048 5.8 -> 6.8).
#include "gemm_direct_kernel.h"

bool gemm_direct_conv_fits(int M, int N, int K, int col, int channels, int taps) {
  return M >= 1 && M <= 16 && !layout_wide(N, K) && K > 0 && K % 8 == 0 && N % 4 == 0 && taps == 4 &&
         gemm_direct_columns(M, N) >= 8 && col % 4 == 0 && channels % 4 == 0 && channels > 0 &&
         col >= 0 && col + channels <= N;
}

int gemm_direct_conv(const ConvArgs& a, hipStream_t stream) {
  const bool deep = layout_deep(a.N, a.K), narrow = gemm_direct_columns(a.M, a.N) == 8;
  TS_DIRECT_ROWS(a.M, {
    if (deep && narrow) launch<1, 8, float, false, false, 4, 4, false, false, 8, AR, true>(a, stream);
    else if (deep) launch<1, 8, float, false, false, 4, 4, false, false, 16, AR, true>(a, stream);
    else if (narrow) launch<1, 4, float, false, false, 4, 4, false, false, 8, AR, true>(a, stream);
    else launch<1, 4, float, false, false, 4, 4, false, false, 16, AR, true>(a, stream);
  })
  return 0;
}

extern "C" int ts_gemm_conv_fits(int M, int N, int K, int col, int channels, int taps) {
  return gemm_direct_conv_fits(M, N, K, col, channels, taps);
}

// C [M, N] float32 = a w^T (bfloat16), out [M, channels] the convolution (as ts_conv_silu's) of its
// columns [col, col + channels); row m is the token at positions[m] of the request in slot
// slot_ids[m], whose last inputs are in `state` [slots, 3, channels].
extern "C" int ts_gemm_conv_silu(const void* a, const void* w, float* c, int M, int N, int K, int col,
                                 int channels, int taps, const float* conv_w, const float* bias,
                                 const float* in_bias, float* state, float* out,
                                 const int* positions, const int* slot_ids, int plain,
                                 hipStream_t stream) {
  if (M <= 0) return 0;
  if (!gemm_direct_conv_fits(M, N, K, col, channels, taps))
    TS_FAIL("gemm_conv_silu: %d rows, weight [%d, %d], %d channels of %d taps from column %d are not taken",
            M, N, K, channels, taps, col);
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)conv_w | (uintptr_t)bias | (uintptr_t)in_bias |
       (uintptr_t)state | (uintptr_t)out) & 15)
    TS_FAIL("gemm_conv_silu: operands must be 16-byte aligned");
  ConvArgs d = {};
  d.A = (const bf16_t*)a, d.W = (const bf16_t*)w, d.C = c, d.M = M, d.N = N, d.K = K;
  d.conv_w = conv_w, d.conv_b = bias, d.conv_in_b = in_bias, d.conv_state = state, d.conv_out = out;
  d.conv_pos = positions, d.conv_slots = slot_ids;
  d.conv_col = col, d.conv_channels = channels, d.conv_plain = plain;
  if (gemm_direct_conv(d, stream)) return -1;
  TS_CHECK_LAUNCH("gemm_conv_silu");
  return 0;
}
