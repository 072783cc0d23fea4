// The recurrences of matrix_state.hip and ssm.hip for steps in which every entry brings one
// token, as decode steps are: S <- g S + k u^T, o = S^T q, once.
//
// What bounds such a step is the state, read and written once: 16 heads of 128 x 128 and 8
// requests are 8.4 MB each way.  The kernels that walk an entry's tokens are made for its
// arithmetic: they stage 16 tokens' operands, clear their buffers and wait at barriers before
// a token is touched, and read a state an element at a time.  Here a thread asks for its
// operands, then for its rows of the state 16 bytes at a time, and has all of it in flight at
// once; while the state is on its way the operands go to LDS.  Lanes and rows lie as in the
// walk (eight lanes share a column, four columns a thread), and sums are added in its order,
// so the results are the walk's to the bit.
//
// A step of 8 requests, walked and here: fixed decays, 16 heads of 128 x 128, 17.0 and 6.0 us;
// state space, 64 heads of 128 x 64, 15.1 and 9.7 us (33.5 MB: 3.5 TB/s); the delta rule with its
// gates in front and its norm behind, 22.4 us in three kernels and 8.3 in one, with a decay per
// row of 8 heads of 64 x 128 20.4 and 6.0.
#include "recurrence_step.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

static __device__ __forceinline__ float sigmoid_f(float v) { return 1.0f / (1.0f + expf(-v)); }
static __device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }
static __device__ __forceinline__ float softplus_f(float v) { return v > 20.f ? v : log1pf(expf(v)); }

constexpr int kSlices = 8;                 // lanes that share a column
constexpr int kCols = 4;                   // columns a thread owns

// Sum over the eight neighbouring lanes that share a column; every one of them gets it.
__device__ __forceinline__ float sum_slices(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));
  return v;
}

// The value the other lane of a pair of neighbours holds.
__device__ __forceinline__ float swap_pair(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));
}

template <int NI>
__device__ __forceinline__ void read_rows(const float* p, float (&r)[NI]) {
  if constexpr (NI % 4 == 0) {
#pragma unroll
    for (int j = 0; j < NI / 4; ++j) {
      const f32x4 v = ((const f32x4*)p)[j];
#pragma unroll
      for (int c = 0; c < 4; ++c) r[4 * j + c] = v[c];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NI; ++j) r[j] = p[j];
  }
}

// ---------------------------------------------------------------- a matrix per head
// N = 8 NI key channels.  A workgroup has 64 columns of a head of an entry (128 threads), or
// with GATED the whole head of up to 128 columns (two threads a column), whose output it then
// norms and gates.
template <int NI, bool DELTA, bool PER_ROW, bool TURN, typename TO, bool GATED>
__global__ __launch_bounds__(256) void recurrence_step_kernel(RecurrenceStepArgs a) {
  constexpr int N = kSlices * NI;
  // a slice's rows in LDS lie side by side, 16 bytes between slices: the eight reads of an
  // instruction fall into different banks
  constexpr int SP = NI + 4;
  __shared__ __align__(16) float q_s[kSlices * SP], k_s[kSlices * SP], g_s[PER_ROW ? kSlices * SP : 1];
  __shared__ __align__(16) float o_s[GATED ? 128 : 1];
  const int h = blockIdx.x, e = blockIdx.y;
  const int s = threadIdx.x % kSlices, cg = threadIdx.x / kSlices;
  const int p0 = blockIdx.z * (blockDim.x / kSlices * kCols) + cg * kCols;
  const bool live = p0 < a.P;
  const int p = live ? p0 : 0;              // (a column past the last reads the first, stores nothing)
  const int hk = h / (a.heads / a.kv_heads);
  const int pos = a.positions[e];
  float* st = a.state + ((int64_t)a.slot_ids[e] * a.heads + h) * N * a.P + p;
  const float* row = a.x + (int64_t)e * a.ld;
  const int n = threadIdx.x;                // the row of S whose operands this thread stages
  const int at = n / NI * SP + n % NI;

  // operands, then the state: all asked for before the first is used
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  constexpr int kKeep = (N + kWave - 1) / kWave;
  float own[GATED ? kKeep : 1], qv = 0.f, kv = 0.f, gv = 1.f, beta = 0.f, g_all = 1.f;
  float2 turn = make_float2(1.f, 0.f);
  f32x4 gate = {0.f, 0.f, 0.f, 0.f}, weight = gate;
  int lanes = 16, part = 0;
  if constexpr (GATED) {
    // the first wavefront makes q a unit vector, the second k
    const float* v = row + (wave == 0 ? a.q_col : a.k_col) + hk * N;
#pragma unroll
    for (int j = 0; j < kKeep; ++j) own[j] = lane + j * kWave < N ? v[lane + j * kWave] : 0.f;
    beta = a.beta[(int64_t)e * a.ldb + h];
    const int zi = PER_ROW ? h * N + min(n, N - 1) : h;
    gv = a.z[(int64_t)e * a.ldz + zi] + a.dt_bias[zi];
    lanes = a.P <= 64 ? 16 : 32;
    part = min(lane % lanes * 4, a.P - 4);
    gate = *(const f32x4*)(a.gate + (int64_t)e * a.ldgate + h * a.P + part);
    weight = *(const f32x4*)(a.norm_w + part);
  } else {
    if (n < N) {
      qv = row[a.q_col + hk * N + n];
      kv = row[a.k_col + hk * N + n];
      if (TURN && n < a.turn_dims) turn = a.turn[(int64_t)pos * (a.turn_dims / 2) + n / 2];
      if (PER_ROW) gv = a.gates[(int64_t)e * a.ldg + a.heads + h * N + n];
    }
    if (DELTA) beta = a.gates[(int64_t)e * a.ldg + h];
    if (!PER_ROW) g_all = a.gates ? a.gates[(int64_t)e * a.ldg + a.heads + h] : a.decay[h];
  }
  f32x4 u = *(const f32x4*)(row + a.v_col + h * a.P + p);
  // (a new sequence's state is read like any other and dropped: no load hangs on a condition)
  f32x4 S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) S[i] = *(const f32x4*)(st + (int64_t)(s * NI + i) * a.P);

  if constexpr (GATED) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < kKeep; ++j) ss = fmaf(own[j], own[j], ss);
    ss = wave_sum(ss);
    const float q_scale = 1.0f / sqrtf((float)N);
    const float r = (1.0f / sqrtf(ss + 1e-6f)) * (wave == 0 ? q_scale : 1.f);
#pragma unroll
    for (int j = 0; j < kKeep; ++j) {
      const int i = lane + j * kWave;
      if (wave < 2 && i < N) (wave == 0 ? q_s : k_s)[i / NI * SP + i % NI] = own[j] * r;
    }
    beta = sigmoid_f(beta);
    gv = expf(-expf(a.a_log[h]) * softplus_f(gv));
    if (!PER_ROW) g_all = gv;
  } else if constexpr (TURN) {
    // (the partner of a pair is the neighbouring lane's)
    const float sn = n & 1 ? turn.y : -turn.y;
    const float qt = fmaf(swap_pair(qv), sn, qv * turn.x);
    const float kt = a.k_scale * fmaf(swap_pair(kv), sn, kv * turn.x);
    if (n < N) q_s[at] = qt, k_s[at] = kt;
  } else {
    if (n < N) q_s[at] = a.silu ? silu_f(qv) : qv, k_s[at] = a.silu ? silu_f(kv) : kv;
  }
  if (PER_ROW && n < N) g_s[at] = gv;
  if (!GATED && a.silu) {
#pragma unroll
    for (int c = 0; c < kCols; ++c) u[c] = silu_f(u[c]);
  }
  __syncthreads();
  float kr[NI], qr[NI];
  read_rows<NI>(k_s + s * SP, kr);
  read_rows<NI>(q_s + s * SP, qr);
  const bool fresh = pos == 0;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int c = 0; c < kCols; ++c) S[i][c] = fresh ? 0.f : S[i][c];
  if constexpr (DELTA) {
    float gr[NI];
    if constexpr (PER_ROW) read_rows<NI>(g_s + s * SP, gr);
    float pred[kCols][2] = {};
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float g = PER_ROW ? gr[i] : g_all;
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        S[i][c] *= g;
        pred[c][i & 1] = fmaf(S[i][c], kr[i], pred[c][i & 1]);
      }
    }
#pragma unroll
    for (int c = 0; c < kCols; ++c) u[c] = beta * (u[c] - sum_slices(pred[c][0] + pred[c][1]));
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int c = 0; c < kCols; ++c) S[i][c] = fmaf(kr[i], u[c], S[i][c]);
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int c = 0; c < kCols; ++c) S[i][c] = fmaf(g_all, S[i][c], kr[i] * u[c]);
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < NI; ++i) *(f32x4*)(st + (int64_t)(s * NI + i) * a.P) = S[i];
  }
  f32x4 o;
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int i = 0; i < NI; i += 2) {
      a0 = fmaf(S[i][c], qr[i], a0);
      a1 = fmaf(S[i + 1][c], qr[i + 1], a1);
    }
    o[c] = sum_slices(a0 + a1);
  }
  if constexpr (!GATED) {
    if (s == 0 && live) *(f32x4*)(a.out + ((int64_t)e * a.heads + h) * a.P + p) = o;
  } else {
    if (s == 0) *(f32x4*)(o_s + p) = o;
    __syncthreads();
    if (wave != 0) return;
    // the head's norm and gate, as gated_norm.h takes them
    const f32x4 v = *(const f32x4*)(o_s + part);
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float sg = 1.0f / (1.0f + expf(-gate[c]));
      gate[c] = a.act == 0 ? sg : gate[c] * sg;
      ss = fmaf(v[c], v[c], ss);
    }
    if (lanes == 32) ss += __shfl_xor(ss, 16, kWave);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, kWave);
    const float r = 1.0f / sqrtf(ss / (float)a.P + a.eps);
    if (lane >= lanes) return;
    typedef TO out4 __attribute__((ext_vector_type(4)));
    out4 w;
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = from_f32<TO>(v[c] * r * weight[c] * gate[c]);
    *(out4*)((TO*)a.gated + ((int64_t)e * a.heads + h) * a.P + part) = w;
  }
}

static bool rows_built(int N) { return N == 16 || N == 32 || N == 64 || N == 128; }

bool recurrence_step_fits(const RecurrenceStepArgs& a) {
  return rows_built(a.N) && a.P % 4 == 0 && a.ld % 4 == 0 && a.v_col % 4 == 0 &&
         (((uintptr_t)a.x | (uintptr_t)a.state | (uintptr_t)a.out) & 15) == 0;
}

#define TS_STEP_ROWS(N, ...)                              \
  switch (N) {                                            \
    case 16: { constexpr int NI = 2; __VA_ARGS__; } break;  \
    case 32: { constexpr int NI = 4; __VA_ARGS__; } break;  \
    case 64: { constexpr int NI = 8; __VA_ARGS__; } break;  \
    default: { constexpr int NI = 16; __VA_ARGS__; } break; \
  }

void launch_recurrence_step(const RecurrenceStepArgs& a, int num_entries, bool delta, bool per_row,
                            hipStream_t stream) {
  const dim3 grid(a.heads, num_entries, (a.P + 63) / 64), block(128);
  TS_STEP_ROWS(a.N, {
    if (delta && per_row)
      hipLaunchKernelGGL((recurrence_step_kernel<NI, true, true, false, float, false>), grid, block, 0, stream, a);
    else if (delta)
      hipLaunchKernelGGL((recurrence_step_kernel<NI, true, false, false, float, false>), grid, block, 0, stream, a);
    else if (a.turn)
      hipLaunchKernelGGL((recurrence_step_kernel<NI, false, false, true, float, false>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((recurrence_step_kernel<NI, false, false, false, float, false>), grid, block, 0, stream, a);
  })
}

// Whether ts_delta_step takes heads of N key channels and P columns.
extern "C" int ts_delta_step_fits(int N, int P) { return rows_built(N) && (P == 64 || P == 128); }

// The gated delta rule of a step in which entry e brings token e alone, from the convolved rows
// to the gated ones: ts_delta_gates, ts_linear_recurrence and ts_norm_gate (a weight shared by
// the heads) in one kernel, to the bit.  qkv [T, ld] holds q | k (kv_heads x N each) | v (heads x
// P), not written; beta at beta_col of proj, z at z_col of its rows, the gate at gate_col of its.
extern "C" int ts_delta_step(const float* qkv, int ld, const float* proj, int ldp, int beta_col,
                             const float* z, int ldz, int z_col, const float* a_log,
                             const float* dt_bias, const float* gate, int ldgate, int gate_col,
                             const float* norm_w, int act, float eps, float* state, void* out,
                             int out_type, const int* positions, const int* slot_ids,
                             int num_entries, int heads, int kv_heads, int N, int P, int per_row,
                             hipStream_t stream) {
  if (num_entries <= 0) return 0;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || !ts_delta_step_fits(N, P))
    TS_FAIL("delta_step: heads=%d kv_heads=%d dim=%d vdim=%d are not built", heads, kv_heads, N, P);
  const int ng = per_row ? heads * N : heads;
  if (ld < 2 * kv_heads * N + heads * P || beta_col < 0 || beta_col + heads > ldp || z_col < 0 ||
      z_col + ng > ldz || gate_col < 0 || gate_col + heads * P > ldgate || (act != 0 && act != 1))
    TS_FAIL("delta_step: columns outside the rows");
  RecurrenceStepArgs a{};
  a.x = qkv, a.ld = ld, a.q_col = 0, a.k_col = kv_heads * N, a.v_col = 2 * kv_heads * N;
  a.state = state, a.positions = positions, a.slot_ids = slot_ids;
  a.heads = heads, a.kv_heads = kv_heads, a.N = N, a.P = P;
  a.beta = proj + beta_col, a.ldb = ldp, a.z = z + z_col, a.ldz = ldz;
  a.a_log = a_log, a.dt_bias = dt_bias, a.gate = gate + gate_col, a.ldgate = ldgate;
  a.norm_w = norm_w, a.act = act, a.eps = eps, a.gated = out;
  if (!recurrence_step_fits(a) || ldgate % 4 ||
      (((uintptr_t)a.gate | (uintptr_t)norm_w | (uintptr_t)out) & 15))
    TS_FAIL("delta_step: rows must begin on 16 bytes");
  const dim3 grid(heads, num_entries), block(2 * P);
  TS_DISPATCH_TYPE(out_type, TO, TS_STEP_ROWS(N, {
    if (per_row)
      hipLaunchKernelGGL((recurrence_step_kernel<NI, true, true, false, TO, true>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((recurrence_step_kernel<NI, true, false, false, TO, true>), grid, block, 0, stream, a);
  }));
  TS_CHECK_LAUNCH("delta_step");
  return 0;
}

// ---------------------------------------------------------------- state space
// The step of ssm.hip's recurrence.  Thread (cg, s) has rows s, s + 8, ... of four columns, as
// in the walk; a workgroup 64 columns.
template <int NI>
__global__ __launch_bounds__(128) void scan_step_kernel(ScanStepArgs a) {
  constexpr int N = kSlices * NI, SP = NI + 4;
  __shared__ __align__(16) float b_s[kSlices * SP], c_s[kSlices * SP];
  const int h = blockIdx.x, e = blockIdx.y;
  const int s = threadIdx.x % kSlices, cg = threadIdx.x / kSlices;
  const int p0 = (blockIdx.z * (128 / kSlices) + cg) * kCols;
  const bool live = p0 < a.P;
  const int p = live ? p0 : 0;
  const int g = h / (a.heads / a.groups), inner = a.heads * a.P;
  const float* row = a.xbc + (int64_t)e * (inner + 2 * a.groups * N);
  float* st = a.state + ((int64_t)a.slot_ids[e] * a.heads + h) * N * a.P + p;
  const bool fresh = a.positions[e] == 0;
  const int n = threadIdx.x, at = n % kSlices * SP + n / kSlices;
  const float bv = row[inner + g * N + min(n, N - 1)];
  const float cv = row[inner + (a.groups + g) * N + min(n, N - 1)];
  const float dt = a.dt[(int64_t)e * a.ldt + h] + a.dt_bias[h];
  const float a_log = a.a_log[h], skip = a.d_skip[h];
  const f32x4 x = *(const f32x4*)(row + h * a.P + p);
  f32x4 S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) S[i] = *(const f32x4*)(st + (int64_t)(s + kSlices * i) * a.P);
  if (n < N) b_s[at] = bv, c_s[at] = cv;
  const float d = softplus_f(dt), decay = expf(-expf(a_log) * d);
  __syncthreads();
  float br[NI], cr[NI];
  read_rows<NI>(b_s + s * SP, br);
  read_rows<NI>(c_s + s * SP, cr);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      S[i][c] = fmaf(decay, fresh ? 0.f : S[i][c], br[i] * (d * x[c]));
      acc[c] = fmaf(S[i][c], cr[i], acc[c]);
    }
    if (live) *(f32x4*)(st + (int64_t)(s + kSlices * i) * a.P) = S[i];
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c) acc[c] = fmaf(skip, x[c], sum_slices(acc[c]));
  if (s == 0 && live) *(f32x4*)(a.y + (int64_t)e * inner + h * a.P + p) = acc;
}

bool scan_step_fits(const ScanStepArgs& a) {
  const int channels = a.heads * a.P + 2 * a.groups * a.N;
  return rows_built(a.N) && a.P % 4 == 0 && channels % 4 == 0 &&
         (((uintptr_t)a.xbc | (uintptr_t)a.state | (uintptr_t)a.y) & 15) == 0;
}

void launch_scan_step(const ScanStepArgs& a, int num_entries, hipStream_t stream) {
  const dim3 grid(a.heads, num_entries, (a.P + 63) / 64);
  TS_STEP_ROWS(a.N, hipLaunchKernelGGL(scan_step_kernel<NI>, grid, dim3(128), 0, stream, a))
}
