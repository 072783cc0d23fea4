// The second steps of two low-rank projections in one launch: out_a [M, Na] = bfloat16(x[:, col_a ..
// + Ka]) Wa^T and out_g [M, Ng] likewise, float32, from the first steps' columns of the float32 rows x.
// A wavefront makes 16 rows by 16 columns on the matrix cores, its operands cut out of x as they
// are read.  Bound by its launch for a few rows and by the outputs' way to memory for many: as two
// copies of columns and two products, for 512 + 1,024 columns of rank 64, it was four launches: 16.5
// us of a decode step of 8 rows, 22.5 of a prompt of 2,048; the step 585 -> 573 us with two such
// layers, the prompt 3,536 -> 3,524.
#include "common.h"

typedef __bf16 bf16x8_lr __attribute__((ext_vector_type(8)));
typedef float f32x4_lr __attribute__((ext_vector_type(4)));

struct LowRankArgs {
  const float* x;
  int ld, M, wide;               // wide: x's pieces of four begin on 16 bytes
  const bf16_t* w[2];            // [n, k]
  float* out[2];                 // [M, n]
  int col[2], n[2], k[2];
  int blocks;                    // of 64 columns of the first
};

__global__ __launch_bounds__(256) void low_rank_pair_kernel(LowRankArgs a) {
  const int which = (int)blockIdx.x >= a.blocks, block = blockIdx.x - (which ? a.blocks : 0);
  const int lane = threadIdx.x % kWave, l = lane % 16, g = lane / 16;
  const int K = a.k[which], N = a.n[which];
  const int n0 = block * 64 + threadIdx.x / kWave * 16, m = blockIdx.y * 16 + l;
  if (n0 >= N) return;
  const float* x = a.x + (int64_t)min(m, a.M - 1) * a.ld + a.col[which] + 8 * g;
  const bf16_t* w = a.w[which] + (int64_t)min(n0 + l, N - 1) * K + 8 * g;
  f32x4_lr sum = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < K; k += 32) {
    float v[8];
    if (a.wide) {
      *(f32x4_lr*)v = *(const f32x4_lr*)(x + k);
      *(f32x4_lr*)(v + 4) = *(const f32x4_lr*)(x + k + 4);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = x[k + j];
    }
    bf16x8_lr xv;
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[j] = (bf16_t)v[j];
    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_lr*)(w + k), xv, sum, 0, 0, 0);
  }
  if (m >= a.M) return;
  float* out = a.out[which] + (int64_t)m * N + n0 + 4 * g;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n0 + 4 * g + r < N) out[r] = sum[r];
}

extern "C" int ts_low_rank_pair_fits(int ka, int kg) {
  return ka > 0 && kg > 0 && ka % 32 == 0 && kg % 32 == 0;
}

extern "C" int ts_low_rank_pair(const float* x, int ld, int M, int col_a, const void* w_a, int n_a,
                                int k_a, float* out_a, int col_g, const void* w_g, int n_g, int k_g,
                                float* out_g, hipStream_t stream) {
  if (M <= 0) return 0;
  if (!ts_low_rank_pair_fits(k_a, k_g) || n_a <= 0 || n_g <= 0)
    TS_FAIL("low_rank_pair: %d columns of rank %d and %d of %d are not taken", n_a, k_a, n_g, k_g);
  if (col_a < 0 || col_a + k_a > ld || col_g < 0 || col_g + k_g > ld)
    TS_FAIL("low_rank_pair: columns outside the rows");
  if (((uintptr_t)w_a | (uintptr_t)w_g) & 15) TS_FAIL("low_rank_pair: weights must be 16-byte aligned");
  const int rows = (M + 15) / 16;
  if (rows > 65535) TS_FAIL("low_rank_pair: M=%d too large for one launch", M);
  LowRankArgs a = {x, ld, M, ((ld | col_a | col_g) % 4 == 0 && ((uintptr_t)x & 15) == 0) ? 1 : 0,
                   {(const bf16_t*)w_a, (const bf16_t*)w_g}, {out_a, out_g}, {col_a, col_g},
                   {n_a, n_g}, {k_a, k_g}, (n_a + 63) / 64};
  hipLaunchKernelGGL(low_rank_pair_kernel, dim3(a.blocks + (n_g + 63) / 64, rows), dim3(256), 0, stream, a);
  TS_CHECK_LAUNCH("low_rank_pair");
  return 0;
}
