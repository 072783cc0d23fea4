// C[M,N] = A[M,K] * W[N,K]^T in float32: float32 operands (bfloat16 ones are widened), float32
// products and sums, no reduced-precision mode.  This is the product of the float32 path and of
// any bfloat16 run whose weights are held in 32-bit; where both operands are float32 and K is a
// multiple of 64, gemm_f32_split.hip takes it.
//
// Every output element adds its K products in an order fixed by K alone, so its value does not
// depend on which other rows are in the call nor on the kernel that the number of rows chooses.
// Where K is a multiple of 4: K is cut into steps of 16, four of them a stretch, the stretches into
// eight runs of equal length.  A step is four float32 matrix-core products
// (v_mfma_f32_16x16x4_f32; elements 4 g + r, g = 0..3, in product r) in two chains from zero, the
// even and the odd r; a run adds the steps' sums in order, the result the sums of pairs of runs in
// order.  Chains of eight products and not of a stretch's 64, because their roundings are what an
// element's error mostly is: 9.6e-8 of the result at K = 1,024 against 1.58e-7, 1.1e-7 against
// 1.6e-7 at 2,048, for 4 to 10 % of the tiles' time.  Another K adds in index order in one accumulator.
#include <type_traits>

#include "common.h"
#include "gemm_f32_split.h"

constexpr int kTile = 64;   // output tile edge per workgroup
constexpr int kStep = 16;   // K elements staged per iteration

template <typename TA, typename TW, typename TC>
__global__ __launch_bounds__(256) void gemm_fma_kernel(const TA* __restrict__ A,
                                                       const TW* __restrict__ W,
                                                       TC* __restrict__ C, int M, int N, int K) {
  __shared__ float As[kStep][kTile + 4];
  __shared__ float Ws[kStep][kTile + 4];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const int64_t m0 = (int64_t)blockIdx.y * kTile, n0 = (int64_t)blockIdx.x * kTile;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += kStep) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int idx = tid + r * 256;
      const int row = idx / kStep, k = idx % kStep;
      const bool kin = k0 + k < K;
      As[k][row] = (kin && m0 + row < M) ? to_f32(A[(m0 + row) * K + k0 + k]) : 0.f;
      Ws[k][row] = (kin && n0 + row < N) ? to_f32(W[(n0 + row) * K + k0 + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kStep; ++k) {
      float a[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = Ws[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = n0 + tx * 4 + j;
      if (n < N) C[m * N + n] = from_f32<TC>(acc[i][j]);
    }
  }
}

// ---------------------------------------------------------------- K a multiple of 4
// Matrix operands: lane (g, l) = (lane / 16, lane % 16) holds row l of A or W, elements
// 4 g .. 4 g + 3 of a step, and rows 4 g + r, column l of the sums.
typedef __attribute__((ext_vector_type(4))) float f32x4_fma;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_fma;
__device__ __forceinline__ f32x4_fma load4_fma(const float* p) { return *(const f32x4_fma*)p; }
__device__ __forceinline__ f32x4_fma load4_fma(const bf16_t* p) {
  const bf16x4_fma v = *(const bf16x4_fma*)p;
  return f32x4_fma{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

constexpr int kRuns = 8, kStretch = 4;     // runs of K, steps of a stretch

// Stretches of a run: the last runs may be shorter or empty.
__host__ __device__ __forceinline__ int stretches_of_run(int K) {
  const int stretches = (K + 16 * kStretch - 1) / (16 * kStretch);
  return (stretches + kRuns - 1) / kRuns;
}

// Few rows (up to 16 MT): a workgroup takes 16 columns, each of its eight wavefronts a run of K, so
// a weight is read once, straight into the matrix cores' operands, a stretch ahead of its use.
// Bound by the rate at which a compute unit takes load instructions: one of W and MT of A
// (cached) a step.
template <typename TA, typename TW, typename TC, int MT>
__global__ __launch_bounds__(kRuns* kWave) void gemm_f32_rows_kernel(
    const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N, int K) {
  __shared__ __align__(16) float part[kRuns][MT][256];
  const int run = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int l = lane % 16, g = lane / 16;
  const int64_t n0 = (int64_t)blockIdx.x * 16;
  const int steps = (K + 15) / 16, per = stretches_of_run(K) * kStretch;
  const int begin = run * per, end = min(begin + per, steps);
  const TW* w_row = W + min(n0 + l, (int64_t)N - 1) * K + 4 * g;
  const TA* a_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = A + (int64_t)min(16 * i + l, M - 1) * K + 4 * g;
  const f32x4_fma zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_fma sum[MT], w[2][kStretch], a[2][kStretch][MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) sum[i] = zero;
  auto fetch = [&](int half, int step0) {
#pragma unroll
    for (int u = 0; u < kStretch; ++u) {
      // (a step behind the run is read from the run's last place and not used)
      const int k = min(min(step0 + u, end - 1) * 16, K - 4 - 4 * g);
      w[half][u] = load4_fma(w_row + k);
#pragma unroll
      for (int i = 0; i < MT; ++i) a[half][u][i] = load4_fma(a_row[i] + k);
    }
  };
  auto multiply = [&](int half, int step0) {
#pragma unroll
    for (int u = 0; u < kStretch; ++u) {
      if (step0 + u >= end) break;
      const bool inside = (step0 + u) * 16 + 4 * g < K;      // (K's last step may be cut)
      const f32x4_fma wv = inside ? w[half][u] : zero;
      f32x4_fma chain[MT][2];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          chain[i][r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              inside ? a[half][u][i][r] : 0.f, wv[r], r < 2 ? zero : chain[i][r & 1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MT; ++i) sum[i] += chain[i][0] + chain[i][1];
    }
  };
  if (begin < end) {
    fetch(0, begin);
    for (int s = begin; s < end; s += 2 * kStretch) {
      if (s + kStretch < end) fetch(1, s + kStretch);
      multiply(0, s);
      if (s + kStretch >= end) break;
      if (s + 2 * kStretch < end) fetch(0, s + 2 * kStretch);
      multiply(1, s + kStretch);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) *(f32x4_fma*)&part[run][i][lane * 4] = sum[i];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * 256; e += kRuns * kWave) {
    const int i = e / 256, row = e % 256 / 16, col = e % 16;
    const int at = (row / 4 * 16 + col) * 4 + row % 4;
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < kRuns; r += 2) v += part[r][i][at] + part[r + 1][i][at];
    const int m = 16 * i + row;
    if (m < M && n0 + col < N) C[(int64_t)m * N + n0 + col] = from_f32<TC>(v);
  }
}

// Many rows: a BM x BN tile a workgroup.  Its wavefronts stand in G groups of four, a group takes
// 8 / G runs of K, a wavefront a quarter of the tile, operands through two LDS buffers of KS
// elements of K a group, those of the turn after the next on their way in registers.  The float32 matrix rate (256
// operations a cycle and unit) is low enough that LDS and memory keep up with any tile; what
// counts is that tiles fill the units and that a SIMD has wavefronts enough to hide the trips to
// LDS and memory, so small products take small tiles and more groups (o and down of the 0.6B
// shape, 501 rows: 43 us with one group of a 32 x 64 tile, which is as long with 130 rows).
template <typename TA, typename TW, typename TC, int BM, int BN, int KS, int G>
__global__ __launch_bounds__(256 * G, BM == 32 ? 4 : BM == 64 ? (KS == 32 ? 3 : 2) : 1) void gemm_f32_tile_kernel(
    const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N, int K) {
  constexpr int TM = BM / 32, TN = BN / 32, LD = KS + 4, Q = KS / 4, ROWS = BM + BN;
  constexpr int COUNT = ROWS * Q / 256, STEP = 256 / Q, OWN = kRuns / G;
  constexpr int STEPS = KS / 16, TURNS = kStretch / STEPS;       // steps a turn, turns a stretch
  static_assert(ROWS * Q % 256 == 0 && 256 % Q == 0 && BM % STEP == 0, "whole rows a turn");
  static_assert(STEPS % 2 == 0 && kStretch % STEPS == 0, "operands in two sets by turns");
  static_assert(G == 1 || OWN == 2, "a group's runs are one pair, or it has all of them");
  extern __shared__ __align__(16) float lds[];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256), tid = threadIdx.x % 256;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int l = lane % 16, g = lane / 16, wm = wave / 2, wn = wave % 2;
  const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;
  const int per = stretches_of_run(K);
  const f32x4_fma zero = {0.f, 0.f, 0.f, 0.f};
  const int row0 = tid / Q;
  // (a group's part of K; what lies behind K is zeros, which change no sum)
  int k = group * OWN * per * 16 * kStretch + tid % Q * 4;
  float* buffers = lds + group * 2 * ROWS * LD;
  f32x4_fma next[COUNT];
  auto fetch = [&] {
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const int row = row0 + u * STEP;     // of A's BM rows, then of W's BN
      next[u] = zero;
      if (k < K) {
        if (u * STEP < BM) next[u] = load4_fma(A + min(m0 + row, (int64_t)M - 1) * K + k);
        else next[u] = load4_fma(W + min(n0 + row - BM, (int64_t)N - 1) * K + k);
      }
    }
    k += KS;
  };
  float* put = buffers + row0 * LD + tid % Q * 4;
  auto commit = [&](int which) {
#pragma unroll
    for (int u = 0; u < COUNT; ++u)
      *(f32x4_fma*)(put + which * ROWS * LD + u * STEP * LD) = next[u];
  };
  fetch();
  commit(0);
  fetch();
  __syncthreads();
  // A step's operands are read from LDS while the step before is multiplied, a turn's first
  // while the last step of the turn before is: the barrier that says that every wavefront has
  // put the next turn's operands down, and has read the last of this one's, stands in front
  // of that step's products.
  f32x4_fma af[2][TM], wf[2][TN];
  const float* a_s = buffers + (wm * 16 * TM + l) * LD + 4 * g;
  const float* w_s = buffers + (BM + wn * 16 * TN + l) * LD + 4 * g;
  auto read = [&](int which, int u) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      af[u & 1][i] = *(const f32x4_fma*)(a_s + which * ROWS * LD + 16 * u + 16 * i * LD);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      wf[u & 1][j] = *(const f32x4_fma*)(w_s + which * ROWS * LD + 16 * u + 16 * j * LD);
  };
  read(0, 0);
  int which = 0;
  // A row of tiles is multiplied while the row before is added to its run.
  f32x4_fma chain[2][TN][2], run[TM][TN], pair[TM][TN], all[TM][TN];
  auto add = [&](int row, int set) {
#pragma unroll
    for (int j = 0; j < TN; ++j) run[row][j] += chain[set][j][0] + chain[set][j][1];
  };
  auto turn = [&] {
    commit(which ^ 1);
    fetch();
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      if (u + 1 < STEPS) {
        read(which, u + 1);
      } else {
        __syncthreads();
        which ^= 1;
        read(which, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int set = (u * TM + i) & 1;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            chain[set][j][r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                af[u & 1][i][r], wf[u & 1][j][r], r < 2 ? zero : chain[set][j][r & 1], 0, 0, 0);
        add(i > 0 ? i - 1 : TM - 1, set ^ 1);
        // (the additions in the products' shadow, from the fourth product on, when the last ones
        // of the row before have ended)
        __builtin_amdgcn_sched_group_barrier(8, 3, 0);
#pragma unroll
        for (int m = 3; m < 4 * TN; ++m) {
          __builtin_amdgcn_sched_group_barrier(8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(2, TN == 2 ? 4 : 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto clear = [&](f32x4_fma (&sums)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[i][j] = zero;
  };
  auto gather = [&](f32x4_fma (&sums)[TM][TN], const f32x4_fma (&more)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[i][j] += more[i][j];
  };
  clear(all);
  // (of one group, runs behind K are left out; several meet at the same barriers and make theirs)
  auto there = [&](int own) { return G > 1 || own * per * 16 * kStretch < K; };
#pragma unroll 1
  for (int o = 0; o < OWN && there(o); o += 2) {
    clear(pair);
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      clear(run);
#pragma unroll
      for (int j = 0; j < TN; ++j) chain[1][j][0] = chain[1][j][1] = zero;
#pragma unroll 1
      for (int t = 0; t < per * TURNS; ++t) turn();
      add(TM - 1, 1);
      gather(pair, run);
    }
    gather(all, pair);
  }
  __syncthreads();
  if (G > 1) {
    // the other groups' pair of runs through LDS, [group - 1][wave][tile][lane]
    auto at = [&](int gr, int i, int j) {
      return (f32x4_fma*)(lds + ((((gr - 1) * 4 + wave) * TM + i) * TN + j) * 256 + lane * 4);
    };
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *at(group, i, j) = all[i][j];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        for (int gr = 1; gr < G; ++gr) all[i][j] += *at(gr, i, j);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + (wm * TM + i) * 16 + 4 * g + r, n = n0 + (wn * TN + j) * 16 + l;
        if (m < M && n < N) C[m * N + n] = from_f32<TC>(all[i][j][r]);
      }
}

template <typename TA, typename TW, typename TC, int BM, int BN, int KS, int G>
static int launch_tile(const TA* A, const TW* W, TC* C, int M, int N, int K, hipStream_t stream) {
  constexpr int operands = G * 2 * (BM + BN) * (KS + 4), sums = (G - 1) * BM * BN;
  const size_t lds = (size_t)(operands > sums ? operands : sums) * sizeof(float);
  auto* fn = gemm_f32_tile_kernel<TA, TW, TC, BM, BN, KS, G>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return -1;
  hipLaunchKernelGGL(fn, dim3((N + BN - 1) / BN, (M + BM - 1) / BM), dim3(256 * G), lds, stream, A, W, C, M, N, K);
  return 0;
}

template <typename TA, typename TW, typename TC>
static int launch_f32(const TA* A, const TW* W, TC* C, int M, int N, int K, hipStream_t stream) {
  if constexpr (std::is_same_v<TA, float> && std::is_same_v<TW, float> && std::is_same_v<TC, float>) {
    if (gemm_f32_split_fits(K)) return gemm_f32_split_launch(A, W, C, M, N, K, 0, stream);
  }
  const dim3 block(kRuns * kWave), grid((N + 15) / 16);
  if (M <= 16) {
    hipLaunchKernelGGL((gemm_f32_rows_kernel<TA, TW, TC, 1>), grid, block, 0, stream, A, W, C, M, N, K);
    return 0;
  }
  if (M <= 32) {
    hipLaunchKernelGGL((gemm_f32_rows_kernel<TA, TW, TC, 2>), grid, block, 0, stream, A, W, C, M, N, K);
    return 0;
  }
  if (M <= 64) {
    hipLaunchKernelGGL((gemm_f32_rows_kernel<TA, TW, TC, 4>), grid, block, 0, stream, A, W, C, M, N, K);
    return 0;
  }
  // the largest tile that still gives every unit one
  auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (tiles(128, 128) >= 256) return launch_tile<TA, TW, TC, 128, 128, 32, 1>(A, W, C, M, N, K, stream);
  // (64 x 64: half as many turns, or the third workgroup of a unit where there is one: 512 and 768
  // tiles of K = 1,024 54.5 and 84.0 us with turns of 64, 54.6 and 78.1 with turns of 32; 256 of
  // K = 8,192 232 and 246)
  if (tiles(64, 64) > 512) return launch_tile<TA, TW, TC, 64, 64, 32, 1>(A, W, C, M, N, K, stream);
  if (tiles(64, 64) >= 256) return launch_tile<TA, TW, TC, 64, 64, 64, 1>(A, W, C, M, N, K, stream);
  return launch_tile<TA, TW, TC, 32, 64, 32, 4>(A, W, C, M, N, K, stream);
}

extern "C" int ts_gemm_fma(const void* a, int a_type, const void* w, int w_type, void* c,
                           int c_type, int M, int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0) TS_FAIL("gemm: K=%d", K);
  // rows of 4 elements must start on 16 (float32) or 8 (bfloat16) bytes for these kernels
  // (a property of K and of the buffers, not of M: which kernel serves a weight never
  // depends on the number of rows)
  const bool rows_ok = K % 4 == 0 && (((uintptr_t)a | (uintptr_t)w) & 15) == 0 && (M + 31) / 32 <= 65535;
  if (rows_ok) {
    int rc = 0;
    TS_DISPATCH_TYPE(a_type, TA, TS_DISPATCH_TYPE(w_type, TW, TS_DISPATCH_TYPE(c_type, TC,
        rc = launch_f32<TA, TW, TC>((const TA*)a, (const TW*)w, (TC*)c, M, N, K, stream))));
    if (rc != 0) TS_FAIL("gemm: a tile needs more LDS than the device gives");
    TS_CHECK_LAUNCH("gemm_fma");
    return 0;
  }
  dim3 grid((N + kTile - 1) / kTile, (M + kTile - 1) / kTile);
  if (grid.y > 65535) TS_FAIL("gemm: M=%d too large for one launch", M);
  TS_DISPATCH_TYPE(a_type, TA, TS_DISPATCH_TYPE(w_type, TW, TS_DISPATCH_TYPE(c_type, TC,
      hipLaunchKernelGGL((gemm_fma_kernel<TA, TW, TC>), grid, dim3(256), 0, stream,
                         (const TA*)a, (const TW*)w, (TC*)c, M, N, K))));
  TS_CHECK_LAUNCH("gemm_fma");
  return 0;
}
