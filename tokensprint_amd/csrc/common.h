// Shared device helpers and the C interface conventions of the kernel library.
//
// Every entry point is `extern "C" int ts_<name>(..., hipStream_t stream)`: it checks
// its arguments on the host, launches on the given stream and returns 0, or returns a
// negative code after storing a message that ts_last_error() hands out.  Element types
// travel as codes: 0 = float32, 1 = bfloat16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#define TS_F32 0
#define TS_BF16 1

typedef __bf16 bf16_t;

extern "C" const char* ts_last_error();
void ts_set_error(const char* fmt, ...);

#define TS_FAIL(...)            \
  do {                          \
    ts_set_error(__VA_ARGS__);  \
    return -1;                  \
  } while (0)

#define TS_CHECK_LAUNCH(name)                                                   \
  do {                                                                          \
    hipError_t e_ = hipGetLastError();                                          \
    if (e_ != hipSuccess) TS_FAIL("%s: launch failed: %s", name, hipGetErrorString(e_)); \
  } while (0)

// Compute units of the current device (256 where it cannot be asked).
inline int compute_units() {
  static int units[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
  if (units[device] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0)
      n = 256;
    units[device] = n;
  }
  return units[device];
}

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16_t x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) { return (bf16_t)x; }

constexpr int kWave = 64;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}

// Sum over a block of up to 1024 threads; every thread gets the result.  `scratch`
// holds one float per wave.  The order of the additions is fixed by the thread layout,
// so a row's result does not depend on what else is in the launch.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < nwaves; ++w) total += scratch[w];
  return total;
}

// Division by a number that the host knows (the compiler's takes 40 instructions).
inline unsigned inverse32(unsigned d) { return d <= 1 ? 0xffffffffu : (unsigned)((1ull << 32) / d); }
// n / d for any n, with inv = inverse32(d): the estimate is at most one short.
__device__ __forceinline__ unsigned divided(unsigned n, unsigned d, unsigned inv) {
  const unsigned q = __umulhi(n, inv);
  return q + (n - q * d >= d ? 1u : 0u);
}

// The same of several sums at once.  `scratch`: N floats per wave.
template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N], float* scratch) {
#pragma unroll
  for (int n = 0; n < N; ++n) v[n] = wave_sum(v[n]);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  __syncthreads();
  if (lane == 0) {
#pragma unroll
    for (int n = 0; n < N; ++n) scratch[N * wave + n] = v[n];
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < N; ++n) v[n] = 0.f;
  for (int w = 0; w < nwaves; ++w) {
#pragma unroll
    for (int n = 0; n < N; ++n) v[n] += scratch[N * w + n];
  }
}

// A thread's share of a row that a workgroup keeps in registers: eight elements, number k at `at(k)`.
// QUADS: two fours side by side, moved 16 (bfloat16: 8) bytes at a time, for rows of a multiple of four
// elements whose operands begin on 16 bytes; else an element at a time, a workgroup's threads apart (8 rows of
// 1,001: the add of a normed row 4.8 us with a row's operands under one condition an element, 5.0 with one each,
// 3.6 with none; the bigram embedding 4.7, 5.9, 3.7).
constexpr int kRowItems = 8;

template <bool QUADS>
struct RowShare {
  int width;
  __device__ __forceinline__ int at(int k) const {
    return QUADS ? ((int)threadIdx.x + k / 4 * (int)blockDim.x) * 4 + k % 4 : (int)threadIdx.x + k * (int)blockDim.x;
  }
  __device__ __forceinline__ bool has(int k) const { return at(k) < width; }
  // (zeros behind the row's end, or where there is nothing to read)
  template <typename T>
  __device__ __forceinline__ void load(const T* row, float (&v)[kRowItems], bool there = true) const {
    if constexpr (QUADS) {
      typedef T four __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int k = 0; k < kRowItems; k += 4) {
        four x = {};
        if (there && has(k)) x = *(const four*)(row + at(k));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[k + j] = to_f32(x[j]);
      }
    } else if (there) {
      // (no load under a condition of its own: behind the row's end its last element again, dropped)
      T x[kRowItems];
#pragma unroll
      for (int k = 0; k < kRowItems; ++k) x[k] = row[min(at(k), width - 1)];
#pragma unroll
      for (int k = 0; k < kRowItems; ++k) v[k] = has(k) ? to_f32(x[k]) : 0.f;
    } else {
#pragma unroll
      for (int k = 0; k < kRowItems; ++k) v[k] = 0.f;
    }
  }
  template <typename T>
  __device__ __forceinline__ void store(T* row, const float (&v)[kRowItems]) const {
    typedef T four __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int k = 0; k < kRowItems; k += QUADS ? 4 : 1) {
      if (!has(k)) continue;
      if constexpr (QUADS) {
        four x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = from_f32<T>(v[k + j]);
        *(four*)(row + at(k)) = x;
      } else {
        row[at(k)] = from_f32<T>(v[k]);
      }
    }
  }
};

// Whether rows of `width` elements of these operands (null or not) can be moved in fours.
template <typename... P>
inline bool rows_in_fours(int width, P... operand) {
  return width % 4 == 0 && (((uintptr_t)operand | ...) & 15) == 0;
}

// 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3))), the tanh form of GELU.
__device__ __forceinline__ float gelu_tanh(float z) {
  return 0.5f * z * (1.0f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
}

// A gated feed-forward's unit, from the results of its two products (rounded to the
// activation type first wherever a product makes it in its epilogue, as the path through
// memory stores them): silu(gate) * up, or, with a
// positive limit, g sigmoid(1.702 g) (u + 1) of g = min(gate, limit) and u = up held
// between -limit and limit, or, with a negative limit, gelu_tanh(gate) * up.
__device__ __forceinline__ float gated_unit(float gate, float up, float limit) {
  if (limit > 0.f) {
    const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
    return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
  }
  if (limit < 0.f) return gelu_tanh(gate) * up;
  return gate / (1.f + expf(-gate)) * up;
}

// Dispatch a two-way element type code to a template argument.
#define TS_DISPATCH_TYPE(code, T, ...)                    \
  if ((code) == TS_F32) { typedef float T; __VA_ARGS__; } \
  else if ((code) == TS_BF16) { typedef bf16_t T; __VA_ARGS__; } \
  else TS_FAIL("unknown element type code %d", (int)(code));
