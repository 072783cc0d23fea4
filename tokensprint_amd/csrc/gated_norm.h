// Parts of rows, each divided by its own root mean square and gated, for the mixers whose output
// is: y / rms(y) * w * act(gate) (GATE_FIRST false), or v / rms(v) * w of v = y * act(gate) (true).
#pragma once
#include "common.h"

// A row of `rows` has `groups` parts of `size` columns (a multiple of 4); y [rows, groups * size],
// gate columns [gate_col, gate_col + groups * size) of rows of ldgate; w: `size` values shared by
// the parts, groups * size of them, or null.  act 0: sigmoid, 1: SiLU.
struct GatedNormArgs {
  const float *y, *gate, *w;
  void* out;
  int64_t units;            // rows * groups
  int ldgate, gate_col, w_shared, size, groups, act;
  float eps;
};

// LANES neighbouring lanes take a part, QUADS times four columns each, all of its operands asked
// for at once; LANES 256: a workgroup, its wavefronts' sums through LDS.  (A wavefront that read
// a part twice, an element a lane and a trip, took 25 us for the parts of 2,048 columns of a
// step of 8 rows as of one of 2,048, and 15 us for 16 parts of 128 of 2,048 rows.)
template <typename TO, bool GATE_FIRST, int LANES, int QUADS>
__global__ __launch_bounds__(256) void gated_norm_kernel(GatedNormArgs a) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  __shared__ float scratch[4];
  const int64_t unit = (int64_t)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  const bool live = unit < a.units;
  const int lane = threadIdx.x % LANES;
  const int64_t row = live ? unit / a.groups : 0;
  const int part = live ? (int)(unit % a.groups) : 0;
  const float* y = a.y + (row * a.groups + part) * a.size;
  const float* gate = a.gate + row * a.ldgate + a.gate_col + part * a.size;
  const float* w = a.w ? a.w + (a.w_shared ? 0 : part * a.size) : nullptr;
  f32x4 v[QUADS], g[QUADS], wt[QUADS];
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    const int i = (lane + q * LANES) * 4;
    v[q] = g[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    wt[q] = f32x4{1.f, 1.f, 1.f, 1.f};
    if (live && i < a.size) {
      v[q] = *(const f32x4*)(y + i);
      g[q] = *(const f32x4*)(gate + i);
      if (w) wt[q] = *(const f32x4*)(w + i);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < QUADS; ++q)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float s = 1.0f / (1.0f + expf(-g[q][j]));
      g[q][j] = a.act == 0 ? s : g[q][j] * s;
      if (GATE_FIRST) v[q][j] *= g[q][j];
      ss = fmaf(v[q][j], v[q][j], ss);
    }
  if (LANES == 256) {
    ss = block_sum(ss, scratch);
  } else {
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
  }
  if (!live) return;
  const float r = 1.0f / sqrtf(ss / (float)a.size + a.eps);
  TO* out = (TO*)a.out + (row * a.groups + part) * a.size;
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    const int i = (lane + q * LANES) * 4;
    if (i >= a.size) continue;
    typedef TO out4 __attribute__((ext_vector_type(4)));
    out4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = from_f32<TO>(GATE_FIRST ? v[q][j] * r * wt[q][j] : v[q][j] * r * wt[q][j] * g[q][j]);
    *(out4*)(out + i) = o;
  }
}

// Whether the kernel above takes these operands: columns in fours on 16 bytes, up to 4,096 a part.
inline bool gated_norm_fits(const GatedNormArgs& a) {
  return a.size % 4 == 0 && a.size <= 4096 && a.ldgate % 4 == 0 && a.gate_col % 4 == 0 &&
         (((uintptr_t)a.y | (uintptr_t)a.gate | (uintptr_t)a.w | (uintptr_t)a.out) & 15) == 0;
}

template <typename TO, bool GATE_FIRST>
void launch_gated_norm(const GatedNormArgs& a, hipStream_t stream) {
#define TS_GATED_NORM(LANES, QUADS)                                                              \
  hipLaunchKernelGGL((gated_norm_kernel<TO, GATE_FIRST, LANES, QUADS>),                          \
                     dim3((unsigned)((a.units + 256 / LANES - 1) / (256 / LANES))), dim3(256), 0, \
                     stream, a)
  if (a.size <= 64) TS_GATED_NORM(16, 1);
  else if (a.size <= 128) TS_GATED_NORM(32, 1);
  else if (a.size <= 256) TS_GATED_NORM(64, 1);
  else if (a.size <= 512) TS_GATED_NORM(64, 2);
  else if (a.size <= 1024) TS_GATED_NORM(256, 1);
  else if (a.size <= 2048) TS_GATED_NORM(256, 2);
  else TS_GATED_NORM(256, 4);
#undef TS_GATED_NORM
}
