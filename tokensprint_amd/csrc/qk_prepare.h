// What the q/k preparation is called with, and a row's pieces of eight elements, for the kernels that
// do it: qk_prepare.hip, and the product that has it in its epilogue (gemm_tiled_heads.hip).
#pragma once
#include "common.h"

struct QkPrepareArgs {
  const void* qkv;       // [T, (nq + 2*nkv) * hd + row_extra]
  void* q_out;           // [T, nq, hd]
  void* k_dst;           // pages [num_pages, nkv, P, hd], or flat [T, nkv, hd] if !paged
  void* v_dst;           // pages [num_pages, nkv, hd, P] (transposed), or flat [T, nkv, hd]
  const float* q_weight; // [hd] or null: no norm
  const float* k_weight;
  const float* cos;      // [max_pos, hd/2] or null: no rotation
  const float* sin;
  const int* positions;      // [T]
  const int* entry_of_token; // [T]
  const int* table;          // [B, table_width]
  int table_width;
  int num_tokens, nq, nkv, hd, page_size, max_pos;
  int paged;             // 1: k_dst/v_dst are cache pages; 0: flat buffers
  int store_kv;          // 0: q only
  float eps;
  int row_extra;         // further columns of a qkv row behind the heads (another product's)
};

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_qk;
typedef __attribute__((ext_vector_type(4))) float f32x4_qk;

// Eight consecutive elements of a row as they are loaded, and as they are stored.
template <typename T>
struct Eight;
template <>
struct Eight<bf16_t> {
  bf16x8_qk x;
  __device__ __forceinline__ void load(const bf16_t* p) { x = *(const bf16x8_qk*)p; }
  __device__ __forceinline__ void store(bf16_t* p) const { *(bf16x8_qk*)p = x; }
  __device__ __forceinline__ float get(int j) const { return (float)x[j]; }
  __device__ __forceinline__ void set(int j, float v) { x[j] = (bf16_t)v; }
};
template <>
struct Eight<float> {
  f32x4_qk lo, hi;
  __device__ __forceinline__ void load(const float* p) { lo = *(const f32x4_qk*)p; hi = *(const f32x4_qk*)(p + 4); }
  __device__ __forceinline__ void store(float* p) const { *(f32x4_qk*)p = lo; *(f32x4_qk*)(p + 4) = hi; }
  __device__ __forceinline__ float get(int j) const { return j < 4 ? lo[j] : hi[j - 4]; }
  __device__ __forceinline__ void set(int j, float v) { if (j < 4) lo[j] = v; else hi[j - 4] = v; }
};

// The factor of a head's norm, from the squares of this lane's eight elements and those of the other
// lanes of its group of `lanes`.
__device__ __forceinline__ float head_rstd(const float (&v)[8], int lanes, int hd, float eps) {
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ss += v[j] * v[j];
  for (int o = 1; o < lanes; o <<= 1) ss += __shfl_xor(ss, o, kWave);
  return rsqrtf(ss / (float)hd + eps);
}

// An element of the first half of a head (or the second) turned with its partner's of the other.
__device__ __forceinline__ float head_turned(float v, float other, float c, float s, bool first) {
  return first ? v * c - other * s : v * c + other * s;
}
