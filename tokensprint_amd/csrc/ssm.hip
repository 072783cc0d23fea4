// Kernels of a selective state-space mixer with one scalar decay per head and token:
// the short causal convolution with SiLU, the recurrence itself, and the gated group norm
// behind it.  All arithmetic in float32; the recurrence's state and the convolution's last
// inputs live in float32 per-request slots and are carried from step to step.
//
// A request's state is read only where a portion does not start at position 0, and is
// written once a portion, by the thread that owns the element.
#include "chunked_state.h"
#include "gated_norm.h"
#include "recurrence_step.h"

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus_f(float v) { return v > 20.f ? v : log1pf(expf(v)); }

// ---------------------------------------------------------------- convolution
// u = rows of `proj` (leading dimension ld) from column `col`, `channels` wide.
// (bias may be null: none.)
// out_t[c] = silu(bias[c] + sum_k w[c][k] * u_(t - (taps-1) + k)[c]); inputs in front of
// the sequence are zero, inputs in front of the portion come from state[slot][taps-1][C],
// whose row j holds the input at position start - (taps-1) + j.

// `in_bias` (may be null): added to every input of the sequence before the convolution (the
// zeros in front of the sequence stay zeros; the state holds inputs with it added).
// `plain` 1: no activation behind the convolution.

// One thread per (token, channel); writes no state.
__global__ __launch_bounds__(256) void conv_silu_kernel(
    const float* __restrict__ proj, int ld, int col, int channels, int taps,
    const float* __restrict__ w, const float* __restrict__ bias, const float* __restrict__ state,
    float* __restrict__ out, BatchView b, int num_tokens, const float* __restrict__ in_bias,
    int plain) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)num_tokens * channels) return;
  const int t = (int)(idx / channels), c = (int)(idx % channels);
  const int e = b.entry_of_token[t];
  const int first = b.q_start[e], pos = b.positions[t];
  const float* st = state + (int64_t)b.slot_ids[e] * (taps - 1) * channels;
  float acc = bias ? bias[c] : 0.f;
  const float ib = in_bias ? in_bias[c] : 0.f;
  for (int k = 0; k < taps; ++k) {
    const int back = taps - 1 - k;
    if (pos - back < 0) continue;
    float v;
    if (t - back >= first) v = proj[(int64_t)(t - back) * ld + col + c] + ib;
    else v = st[(int64_t)(taps - 1 - (first - (t - back))) * channels + c];
    acc = fmaf(w[c * taps + k], v, acc);
  }
  out[(int64_t)t * channels + c] = plain ? acc : silu_f(acc);
}

// The same for long steps: a thread takes kConvRun consecutive tokens of one channel, so an
// input is read once for all the taps that meet it (kept in registers) instead of once a
// tap.  An output's sum runs over the taps in the same order as in the kernel above.
constexpr int kConvRun = 8, kConvMaxTaps = 8;
__global__ __launch_bounds__(256) void conv_silu_run_kernel(
    const float* __restrict__ proj, int ld, int col, int channels, int taps,
    const float* __restrict__ w, const float* __restrict__ bias, const float* __restrict__ state,
    float* __restrict__ out, BatchView b, int num_tokens, const float* __restrict__ in_bias,
    int plain) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int t0 = blockIdx.y * kConvRun;
  const float ib = in_bias ? in_bias[c] : 0.f, bc = bias ? bias[c] : 0.f;
  float wk[kConvMaxTaps], raw[kConvRun + kConvMaxTaps - 1];
#pragma unroll
  for (int k = 0; k < kConvMaxTaps; ++k) wk[k] = w[c * taps + min(k, taps - 1)];
  // raw[j]: the input of flat row t0 - (taps - 1) + j, whatever entry it belongs to (another row's
  // where there is none: no output takes that)
#pragma unroll
  for (int j = 0; j < kConvRun + kConvMaxTaps - 1; ++j)
    raw[j] = proj[(int64_t)min(max(t0 - (taps - 1) + j, 0), num_tokens - 1) * ld + col + c];
#pragma unroll
  for (int j = 0; j < kConvRun + kConvMaxTaps - 1; ++j) raw[j] += ib;
#pragma unroll
  for (int i = 0; i < kConvRun; ++i) {
    const int t = t0 + i;
    if (t >= num_tokens) break;
    const int e = b.entry_of_token[t];
    const int first = b.q_start[e], pos = b.positions[t];
    const float* st = state + (int64_t)b.slot_ids[e] * (taps - 1) * channels;
    float acc = bc;
#pragma unroll
    for (int k = 0; k < kConvMaxTaps; ++k) {
      if (k >= taps) break;
      const int back = taps - 1 - k;
      if (pos - back < 0) continue;
      float v;
      if (t - back >= first) v = raw[i + k];
      else v = st[(int64_t)(taps - 1 - (first - (t - back))) * channels + c];
      acc = fmaf(wk[k], v, acc);
    }
    out[(int64_t)t * channels + c] = plain ? acc : silu_f(acc);
  }
}

// The same with four channels a thread, for up to four taps and rows whose channels lie in fours
// on 16 bytes: loads and stores of 16 bytes, and no look at a token's entry where the thread's
// tokens and the inputs in front of them are one entry's (30 against 39 us for 2,048 tokens of
// 6,144 channels).  Four taps are a channel's 16 bytes: one by one, four of 64 lanes' 256 bytes a load, they
// cost a unit more than the inputs (sixteen loads, each naming 32 lines of 128 bytes; 31.3 -> 27.3 us).  No load
// hangs on a condition (each was waited for before the next was sent; in a prompt's step 27.9 -> 24.2 us, 4,096
// channels 17.7 -> 14.5), and there are no more of them than TAPS taps take (two taps of 6,144 channels 29.4 us
// with those of four, 21.9).
constexpr int kConvRunTaps = 4;
template <int TAPS, bool WIDE>        // WIDE: four taps, and w on 16 bytes
__global__ __launch_bounds__(256) void conv_silu_run4_kernel(
    const float* __restrict__ proj, int ld, int col, int channels, const float* __restrict__ w,
    const float* __restrict__ bias, const float* __restrict__ state, float* __restrict__ out, BatchView b,
    int num_tokens, const float* __restrict__ in_bias, int plain) {
  static_assert(!WIDE || TAPS == 4, "a channel's taps in one load");
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  const int t0 = blockIdx.y * kConvRun;
  constexpr int back0 = TAPS - 1;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // (no load hangs on a condition: what is not there is read from a place that is, and dropped)
  const float* some = proj + col + c;
  f32x4 ib = *(const f32x4*)(in_bias ? in_bias + c : some), bc = *(const f32x4*)(bias ? bias + c : some);
  f32x4 wk[TAPS], raw[kConvRun + back0];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 of;                         // one channel's
    if constexpr (WIDE) {
      of = *(const f32x4*)(w + (int64_t)(c + j) * TAPS);
    } else {
#pragma unroll
      for (int k = 0; k < TAPS; ++k) of[k] = w[(int64_t)(c + j) * TAPS + k];
    }
#pragma unroll
    for (int k = 0; k < TAPS; ++k) wk[k][j] = of[k];
  }
  // raw[j]: the input of flat row t0 - (TAPS - 1) + j, whatever entry it belongs to (another row's
  // where there is none: no output takes that)
#pragma unroll
  for (int j = 0; j < kConvRun + back0; ++j)
    raw[j] = *(const f32x4*)(proj + (int64_t)min(max(t0 - back0 + j, 0), num_tokens - 1) * ld + col + c);
  if (!in_bias) ib = zero;
  if (!bias) bc = zero;
#pragma unroll
  for (int j = 0; j < kConvRun + back0; ++j) raw[j] += ib;
  const int e0 = b.entry_of_token[t0], first0 = b.q_start[e0];
  const bool one = b.entry_of_token[min(t0 + kConvRun, num_tokens) - 1] == e0 && first0 <= t0 - back0;
#pragma unroll
  for (int i = 0; i < kConvRun; ++i) {
    const int t = t0 + i;
    if (t >= num_tokens) break;
    f32x4 acc = bc;
    if (one) {
#pragma unroll
      for (int k = 0; k < TAPS; ++k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = fmaf(wk[k][j], raw[i + k][j], acc[j]);
      }
    } else {
      const int e = b.entry_of_token[t];
      const int first = b.q_start[e], pos = b.positions[t];
      const float* st = state + (int64_t)b.slot_ids[e] * back0 * channels;
#pragma unroll
      for (int k = 0; k < TAPS; ++k) {
        const int back = back0 - k;
        if (pos - back < 0) continue;
        const f32x4 v = t - back >= first
            ? raw[i + k] : *(const f32x4*)(st + (int64_t)(back0 - (first - (t - back))) * channels + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = fmaf(wk[k][j], v[j], acc[j]);
      }
    }
    if (!plain) {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = silu_f(acc[j]);
    }
    *(f32x4*)(out + (int64_t)t * channels + c) = acc;
  }
}

// One thread per (entry, channel): the state after the portion.  Row j takes the input at
// position end - (taps-1) + j: from the portion, from the old state further up (read before
// any row at or above it is written: j ascends), or zero in front of the sequence.
__global__ __launch_bounds__(256) void conv_state_kernel(
    const float* __restrict__ proj, int ld, int col, int channels, int taps,
    float* __restrict__ state, BatchView b, int num_entries, const float* __restrict__ in_bias) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)num_entries * channels) return;
  const int e = (int)(idx / channels), c = (int)(idx % channels);
  const int first = b.q_start[e], n = b.q_start[e + 1] - first;
  const int start = b.positions[first];
  float* st = state + (int64_t)b.slot_ids[e] * (taps - 1) * channels;
  const float ib = in_bias ? in_bias[c] : 0.f;
  constexpr int kAtOnce = 4;          // rows asked for before the first is written
  for (int j0 = 0; j0 < taps - 1; j0 += kAtOnce) {
    float v[kAtOnce];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) {
      const int j = min(j0 + u, taps - 2), p = start + n - (taps - 1) + j;
      v[u] = *(p >= start ? proj + (int64_t)(first + p - start) * ld + col + c
                          : st + (int64_t)(j + n) * channels + c);
      v[u] = p >= start ? v[u] + ib : p >= 0 ? v[u] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u)
      if (j0 + u < taps - 1) st[(int64_t)(j0 + u) * channels + c] = v[u];
  }
}

// One thread per (entry, channel) walks the entry's tokens with the last inputs in
// registers and leaves the state: one kernel for steps of few tokens per entry.
constexpr int kMaxTapsInRegisters = 8;
__global__ __launch_bounds__(256) void conv_silu_walk_kernel(
    const float* __restrict__ proj, int ld, int col, int channels, int taps,
    const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ state,
    float* __restrict__ out, BatchView b, int num_entries, const float* __restrict__ in_bias,
    int plain) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)num_entries * channels) return;
  const int e = (int)(idx / channels), c = (int)(idx % channels);
  const int first = b.q_start[e], end = b.q_start[e + 1];
  const float ib = in_bias ? in_bias[c] : 0.f;
  const int start = b.positions[first];
  float* st = state + (int64_t)b.slot_ids[e] * (taps - 1) * channels;
  float hist[kMaxTapsInRegisters], wk[kMaxTapsInRegisters];
#pragma unroll
  for (int j = 0; j < kMaxTapsInRegisters; ++j) {
    hist[j] = 0.f;
    wk[j] = j < taps ? w[c * taps + j] : 0.f;
    // hist[j], j < taps-1: the input at position start - (taps-1) + j
    if (j < taps - 1 && start - (taps - 1) + j >= 0) hist[j] = st[(int64_t)j * channels + c];
  }
  const float bc = bias ? bias[c] : 0.f;
  for (int t = first; t < end; ++t) {
    const float v = proj[(int64_t)t * ld + col + c] + ib;
    float acc = bc;
#pragma unroll
    for (int k = 0; k < kMaxTapsInRegisters; ++k) {
      if (k < taps - 1) acc = fmaf(wk[k], hist[k], acc);
      else if (k == taps - 1) acc = fmaf(wk[k], v, acc);
    }
    out[(int64_t)t * channels + c] = plain ? acc : silu_f(acc);
#pragma unroll
    for (int k = 0; k < kMaxTapsInRegisters - 1; ++k) {
      if (k < taps - 2) hist[k] = hist[k + 1];
      else if (k == taps - 2) hist[k] = v;
    }
  }
#pragma unroll
  for (int j = 0; j < kMaxTapsInRegisters; ++j)
    if (j < taps - 1) st[(int64_t)j * channels + c] = hist[j];
}

extern "C" int ts_conv_silu(const float* proj, int ld, int col, int channels, int taps,
                            const float* w, const float* bias, float* state, float* out,
                            const int* positions, const int* entry_of_token, const int* q_start,
                            const int* slot_ids, int num_tokens, int num_entries, int max_q_len,
                            const float* in_bias, int plain, hipStream_t stream) {
  if (num_tokens <= 0) return 0;
  if (channels <= 0 || taps < 1 || col < 0 || col + channels > ld)
    TS_FAIL("conv_silu: bad sizes channels=%d taps=%d col=%d ld=%d", channels, taps, col, ld);
  BatchView b{positions, entry_of_token, q_start, slot_ids};
  if (max_q_len <= 4 && taps <= kMaxTapsInRegisters) {
    const int64_t n = (int64_t)num_entries * channels;
    hipLaunchKernelGGL(conv_silu_walk_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       stream, proj, ld, col, channels, taps, w, bias, state, out, b,
                       num_entries, in_bias, plain);
    TS_CHECK_LAUNCH("conv_silu (walk)");
    return 0;
  }
  const bool quads = taps <= kConvRunTaps && channels % 4 == 0 && ld % 4 == 0 && col % 4 == 0 &&
                     (((uintptr_t)proj | (uintptr_t)out | (uintptr_t)state | (uintptr_t)bias |
                       (uintptr_t)in_bias) & 15) == 0;
  if (quads && num_tokens >= 256 && (num_tokens + kConvRun - 1) / kConvRun <= 65535) {
    const bool wide = taps == kConvRunTaps && ((uintptr_t)w & 15) == 0;
    const auto kernel = wide        ? conv_silu_run4_kernel<4, true>
                        : taps == 4 ? conv_silu_run4_kernel<4, false>
                        : taps == 3 ? conv_silu_run4_kernel<3, false>
                        : taps == 2 ? conv_silu_run4_kernel<2, false>
                                    : conv_silu_run4_kernel<1, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((channels / 4 + 255) / 256),
                                    (unsigned)((num_tokens + kConvRun - 1) / kConvRun)),
                       dim3(256), 0, stream, proj, ld, col, channels, w, bias, state, out, b, num_tokens, in_bias,
                       plain);
    TS_CHECK_LAUNCH("conv_silu (runs of four channels)");
  } else if (taps <= kConvMaxTaps && num_tokens >= 256 && (num_tokens + kConvRun - 1) / kConvRun <= 65535) {
    hipLaunchKernelGGL(conv_silu_run_kernel,
                       dim3((unsigned)((channels + 255) / 256), (unsigned)((num_tokens + kConvRun - 1) / kConvRun)),
                       dim3(256), 0, stream, proj, ld, col, channels, taps, w, bias, state, out, b,
                       num_tokens, in_bias, plain);
    TS_CHECK_LAUNCH("conv_silu (runs)");
  } else {
    const int64_t n = (int64_t)num_tokens * channels;
    hipLaunchKernelGGL(conv_silu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       proj, ld, col, channels, taps, w, bias, state, out, b, num_tokens, in_bias, plain);
    TS_CHECK_LAUNCH("conv_silu");
  }
  if (taps > 1) {
    const int64_t m = (int64_t)num_entries * channels;
    hipLaunchKernelGGL(conv_state_kernel, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, stream,
                       proj, ld, col, channels, taps, state, b, num_entries, in_bias);
    TS_CHECK_LAUNCH("conv_state");
  }
  return 0;
}

// ---------------------------------------------------------------- recurrence
// Per head h (group g): d = softplus(dt + dt_bias[h]), a = exp(-exp(A_log[h]) d),
//   S <- a S + (d B_g) x_h^T   (S: N x P),   y_h = S^T C_g + D[h] x_h.
// A workgroup serves one (run of tokens, head, 64 columns of P): a thread keeps eight-strided
// rows of four columns in registers, walks the tokens in order and adds the eight slices of
// a column's dot product through the wavefront.
//
// Steps of few tokens per entry walk each entry whole here; long portions run in chunks of 64
// tokens as products of matrices (chunked_state.hip).
struct ScanArgs {
  const float* xbc;       // [T, channels]: x (heads*P) | B (groups*N) | C (groups*N)
  const float* proj;      // [T, ld]: dt at column dt_col
  const float* dt_bias;   // [heads]
  const float* a_log;     // [heads]
  const float* d_skip;    // [heads]
  float* state;           // [slots, heads, N, P]
  float* y;               // [T, heads*P]
  BatchView b;
  int ld, dt_col, channels, heads, P, N, groups;
};

constexpr int kScanSlices = 8;
constexpr int kScanThreads = 128;          // the walking kernel: 8 slices x 16 groups of columns
constexpr int kScanPerThread = 4;          // columns a thread owns
constexpr int kScanBlockCols = kScanThreads / kScanSlices * kScanPerThread;   // 64
constexpr int kScanStage = 16;             // tokens staged in LDS at a time
static_assert(kScanStage * kScanBlockCols == 8 * kScanThreads, "a stage's x: eight loads a thread");

// Thread (cg, s) = (tid / 8, tid % 8) keeps rows s, s + 8, ... of four columns in registers.
// Sixteen tokens' operands (B, C, the workgroup's columns of x, the step and the decay,
// computed once a token) are staged in LDS by all threads together, then walked in order:
// a token costs a thread 2 NI + 3 LDS reads for 8 NI multiply-adds.
template <int NI>
__global__ __launch_bounds__(kScanThreads) void ssm_scan_kernel(ScanArgs a) {
  extern __shared__ float lds[];
  const int N = a.N;
  float* B_s = lds;                                  // [stage][N]
  float* C_s = B_s + kScanStage * N;                 // [stage][N]
  float* x_s = C_s + kScanStage * N;                 // [stage][64]
  float* d_s = x_s + kScanStage * kScanBlockCols;    // [stage]: step size
  float* a_s = d_s + kScanStage;                     // [stage]: decay
  const int h = blockIdx.x;
  const int s = threadIdx.x % kScanSlices, cg = threadIdx.x / kScanSlices;
  const int col0 = blockIdx.z * kScanBlockCols;
  const int p0 = col0 + cg * kScanPerThread;
  const int g = h / (a.heads / a.groups);
  const int e = blockIdx.y, first = a.b.q_start[e], end = a.b.q_start[e + 1];
  const int inner = a.heads * a.P;
  float* st = a.state + ((int64_t)a.b.slot_ids[e] * a.heads + h) * N * a.P;
  float S[NI][kScanPerThread];
  const bool fresh = a.b.positions[first] == 0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int n = s + kScanSlices * i;
#pragma unroll
    for (int c = 0; c < kScanPerThread; ++c)
      S[i][c] = (!fresh && n < N && p0 + c < a.P) ? st[(int64_t)n * a.P + p0 + c] : 0.f;
  }
  const float decay_rate = -expf(a.a_log[h]);
  const float bias = a.dt_bias[h], skip = a.d_skip[h];
  const int b_col = inner + g * N, c_col = inner + a.groups * N + g * N;

  for (int t0 = first; t0 < end; t0 += kScanStage) {
    const int nt = min(kScanStage, end - t0);
    __syncthreads();                                  // the stage before has been walked
    // Loads in batches of eight, all issued before the first is stored, so that a stage
    // costs a few trips to memory and not one per element.
    {
      const int total = nt * N;
      constexpr int U = 8;
      for (int base = 0; base < total; base += kScanThreads * U) {
        float vb[U], vc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = base + u * kScanThreads + threadIdx.x;
          vb[u] = vc[u] = 0.f;
          if (i < total) {
            const float* row = a.xbc + (int64_t)(t0 + i / N) * a.channels;
            vb[u] = row[b_col + i % N];
            vc[u] = row[c_col + i % N];
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = base + u * kScanThreads + threadIdx.x;
          if (i < total) {
            B_s[i] = vb[u];
            C_s[i] = vc[u];
          }
        }
      }
      float vx[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {         // 16 tokens x 64 columns: eight a thread
        const int i = u * kScanThreads + threadIdx.x;
        const int tt = i / kScanBlockCols, c = i % kScanBlockCols;
        vx[u] = (tt < nt && col0 + c < a.P)
            ? a.xbc[(int64_t)(t0 + tt) * a.channels + h * a.P + col0 + c] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) x_s[u * kScanThreads + threadIdx.x] = vx[u];
    }
    if (threadIdx.x < nt) {
      const float d = softplus_f(a.proj[(int64_t)(t0 + threadIdx.x) * a.ld + a.dt_col + h] + bias);
      d_s[threadIdx.x] = d;
      a_s[threadIdx.x] = expf(decay_rate * d);
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float d = d_s[tt], decay = a_s[tt];
      float dx[kScanPerThread], x[kScanPerThread], acc[kScanPerThread];
#pragma unroll
      for (int c = 0; c < kScanPerThread; ++c) {
        x[c] = x_s[tt * kScanBlockCols + cg * kScanPerThread + c];
        dx[c] = d * x[c];
        acc[c] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int n = s + kScanSlices * i;
        const float Bv = n < N ? B_s[tt * N + n] : 0.f;
        const float Cv = n < N ? C_s[tt * N + n] : 0.f;
#pragma unroll
        for (int c = 0; c < kScanPerThread; ++c) {
          S[i][c] = fmaf(decay, S[i][c], Bv * dx[c]);
          acc[c] = fmaf(S[i][c], Cv, acc[c]);
        }
      }
#pragma unroll
      for (int c = 0; c < kScanPerThread; ++c) {
        acc[c] += __shfl_xor(acc[c], 1, kWave);
        acc[c] += __shfl_xor(acc[c], 2, kWave);
        acc[c] += __shfl_xor(acc[c], 4, kWave);
        if (s == 0 && p0 + c < a.P)
          a.y[(int64_t)(t0 + tt) * inner + h * a.P + p0 + c] = fmaf(skip, x[c], acc[c]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int n = s + kScanSlices * i;
#pragma unroll
    for (int c = 0; c < kScanPerThread; ++c)
      if (n < N && p0 + c < a.P) st[(int64_t)n * a.P + p0 + c] = S[i][c];
  }
}

template <int NI>
static void launch_scan(const ScanArgs& a, int num_entries, hipStream_t stream) {
  const unsigned z = (a.P + kScanBlockCols - 1) / kScanBlockCols;
  const size_t lds = (size_t)(kScanStage * (2 * a.N + kScanBlockCols + 2)) * sizeof(float);
  hipLaunchKernelGGL(ssm_scan_kernel<NI>, dim3(a.heads, num_entries, z), dim3(kScanThreads), lds,
                     stream, a);
}

// `num_chunks` 0: every entry is walked whole.  Else `chunks` [num_chunks, 3] cuts every
// entry into runs of ts_chunk_tokens() tokens, the last one shorter (first, one past the last, entry), in
// order, `entry_chunks` [B + 1] says which are whose, and `scratch` has ts_chunked_scratch
// floats.
extern "C" int ts_ssm_scan(const float* xbc, const float* proj, int ld, int dt_col,
                           const float* dt_bias, const float* a_log, const float* d_skip,
                           float* state, float* y, const int* positions,
                           const int* entry_of_token, const int* q_start, const int* slot_ids,
                           int num_tokens, int num_entries, int max_q_len, int heads, int P,
                           int N, int groups,
                           const int* chunks, const int* entry_chunks, int num_chunks,
                           float* scratch, hipStream_t stream) {
  if (num_tokens <= 0) return 0;
  if (heads <= 0 || P <= 0 || N <= 0 || groups <= 0 || heads % groups)
    TS_FAIL("ssm_scan: bad sizes heads=%d vdim=%d state=%d groups=%d", heads, P, N, groups);
  if (N > kScanSlices * 32) TS_FAIL("ssm_scan: state of %d rows, at most %d are built", N, kScanSlices * 32);
  if (dt_col < 0 || dt_col + heads > ld) TS_FAIL("ssm_scan: dt columns outside the projection");
  const BatchView b{positions, entry_of_token, q_start, slot_ids};
  const int channels = heads * P + 2 * groups * N;
  if (num_chunks > 0) {
    if (!chunks || !entry_chunks || !scratch) TS_FAIL("ssm_scan: chunked without its lists and scratch");
    ChunkedArgs c{};                     // q: C, k: B, v: x times its step size
    c.x = xbc, c.state = state, c.out = y, c.b = b;
    c.ld = channels, c.v_col = 0, c.k_col = heads * P, c.q_col = heads * P + groups * N;
    c.heads = heads, c.kv_heads = groups, c.N = N, c.P = P;
    c.dt = proj + dt_col, c.ldg = ld, c.dt_bias = dt_bias, c.a_log = a_log, c.d_skip = d_skip;
    c.k_scale = 1.f, c.chunks = chunks, c.entry_chunks = entry_chunks;
    c.num_chunks = num_chunks, c.num_entries = num_entries, c.max_len = max_q_len, c.scratch = scratch;
    return launch_chunked(c, stream);
  }
  const ScanStepArgs one{xbc, proj + dt_col, dt_bias, a_log, d_skip, state, y, positions, slot_ids,
                         ld, heads, P, N, groups};
  if (max_q_len == 1 && num_tokens == num_entries && scan_step_fits(one)) {       // a token an entry
    launch_scan_step(one, num_entries, stream);
    TS_CHECK_LAUNCH("ssm_scan (one token)");
    return 0;
  }
  ScanArgs a{xbc, proj, dt_bias, a_log, d_skip, state, y, b, ld, dt_col, channels, heads, P, N, groups};
  const int ni = (N + kScanSlices - 1) / kScanSlices;
  if (ni <= 2) launch_scan<2>(a, num_entries, stream);
  else if (ni <= 4) launch_scan<4>(a, num_entries, stream);
  else if (ni <= 8) launch_scan<8>(a, num_entries, stream);
  else if (ni <= 16) launch_scan<16>(a, num_entries, stream);
  else launch_scan<32>(a, num_entries, stream);
  TS_CHECK_LAUNCH("ssm_scan");
  return 0;
}

// ---------------------------------------------------------------- gate and group norm
// v = y * silu(z) (z: the first `inner` columns of proj); each of `groups` equal parts of
// a row is divided by its own root mean square; out = that * w.  (Sizes and places that
// gated_norm.h does not take.)
template <typename TO>
__global__ __launch_bounds__(256) void gated_group_norm_kernel(
    const float* __restrict__ y, const float* __restrict__ proj, int ld,
    const float* __restrict__ w, TO* __restrict__ out, int inner, int groups, float eps) {
  __shared__ float scratch[16];
  const int64_t t = blockIdx.x;
  const int grp = blockIdx.y, size = inner / groups;
  const float* yr = y + t * inner + grp * size;
  const float* zr = proj + t * ld + grp * size;
  float ss = 0.f;
  for (int i = threadIdx.x; i < size; i += blockDim.x) {
    const float v = yr[i] * silu_f(zr[i]);
    ss += v * v;
  }
  const float r = 1.0f / sqrtf(block_sum(ss, scratch) / (float)size + eps);
  TO* o = out + t * inner + grp * size;
  const float* wr = w + grp * size;
  for (int i = threadIdx.x; i < size; i += blockDim.x)
    o[i] = from_f32<TO>(yr[i] * silu_f(zr[i]) * r * wr[i]);
}

extern "C" int ts_gated_group_norm(const float* y, const float* proj, int ld, const float* w,
                                   void* out, int out_type, int rows, int inner, int groups,
                                   float eps, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (inner <= 0 || groups <= 0 || inner % groups || inner > ld)
    TS_FAIL("gated_group_norm: bad sizes inner=%d groups=%d ld=%d", inner, groups, ld);
  const GatedNormArgs n{y, proj, w, out, (int64_t)rows * groups, ld, 0, 0, inner / groups, groups, 1, eps};
  if (gated_norm_fits(n)) {
    TS_DISPATCH_TYPE(out_type, TO, (launch_gated_norm<TO, true>(n, stream)));
    TS_CHECK_LAUNCH("gated_group_norm");
    return 0;
  }
  TS_DISPATCH_TYPE(out_type, TO,
                   hipLaunchKernelGGL(gated_group_norm_kernel<TO>, dim3(rows, groups), dim3(256),
                                      0, stream, y, proj, ld, w, (TO*)out, inner, groups, eps));
  TS_CHECK_LAUNCH("gated_group_norm");
  return 0;
}
