// C[M,N] = A[M,K] W[N,K]^T in float32 with float32 precision, on the bfloat16 matrix cores, for K a
// multiple of 64.
//
// The splitting of an operand into words of lower precision and their products in descending order
// of size are Dekker's (A floating-point technique for extending the available precision, 1971),
// with bfloat16 words as in Henry, Tang and Heinecke (Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations, 2019).  A float32 number is the exact
// sum of three bfloat16 numbers: a0 = bf16(a), a1 = bf16(a - a0), a2 the rest (both differences are
// exact, and a2 has at most seven bits; below 2^-110 the last bits of a2 are below bfloat16's
// smallest number and are lost).  Of the nine products of a pair's parts six are made: (2,0) (0,2)
// (1,1) (1,0) (0,1) and (0,0).  Of those left out, (1,2) and (2,1) are at most 2^-25 of the pair's
// product each, to either side, (2,2) is far smaller.  (With a1 cut off instead of rounded they were
// up to 2^-24 each, both to the side of the product.)  Products of parts are exact in the matrix
// core, and v_mfma_f32_16x16x32_bf16 adds 32 of them with little more than one rounding, where the
// float32 instruction rounds at every one.  That rounding is to one side (a sum's errors had a mean
// of 0.4 of themselves, the same for all rows, and a model's logits were 20 % further off), so of
// every second 32 of K the negative product is made and subtracted; and (0,0), in whose sum it would
// be largest, is added to the five others' outside the matrix core, to nearest.
// Error, of the result's root mean square in 2^-24, beside chains of eight float32 products
// (gemm_fma.hip): K = 64 0.80 / 1.24, 1,024 1.26 / 1.61, 3,072 1.55 / 2.05, 12,288 2.38 / 3.28.
// A row of a single product, in 2^-24 of it: root mean square 0.43 / 0.43, at most 1.5 / 1.0 (the
// two products left out, where one multiply-add rounds once).
//
// Sums: K is cut into eight runs of whole stretches of 64; a run adds the sums of its 32s (five
// instructions from zero, in the order above, and the sixth's), the result the sums of pairs of runs,
// in order.  Every kernel here adds in that order, so an element depends on neither the other rows
// of a call nor their number.
// Where a result is not finite, it may be because a part was not (infinities, and numbers that
// bfloat16 rounds to one, leave a NaN behind): such an element is made again, in float64 (in
// whatever order, it is infinite only if it has to be), by the wavefront that has it.  501 rows of
// NaN with 6,144 x 1,024 take 1.3 ms instead of 0.05, 2,048 with 4,096 x 4,096 3.7 instead of 0.45 (a
// thread an element, one product after the other: 5.7 and 61).
//
// What bounds it: LDS, the matrix cores (six instructions of 16 cycles for 32 of K against eight of
// 32) and what cuts operands in parts, 5.5 instructions a number, one after the other in most of a
// turn.  501 rows, before (float32 instructions) and now, us: 6,144 x 1,024 71 -> 49, 4,096 x 1,024
// 50 -> 36, 1,024 x 2,048 27 -> 25, 1,024 x 3,072 38 -> 35; 2,048 rows of 4,096 x 4,096 794 -> 409.  (The wavefronts of a SIMD cutting and multiplying in turns, or every one for
// itself without LDS in tiles of 32 x 64, is no faster; nor are float32 instructions with operands
// straight into LDS, 65.9 for the first.)
#include "gemm_f32_split.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr f32x4 kZero = {0.f, 0.f, 0.f, 0.f};
constexpr int kRuns = 8;            // of K
constexpr int kTerms = 6;
constexpr int kSmall = kTerms - 1;  // that are added in the matrix core
// parts of A and W that a term multiplies
constexpr int kPartA[kSmall] = {2, 0, 1, 1, 0}, kPartW[kSmall] = {0, 2, 1, 0, 1};

// Two numbers' parts, packed.
__device__ __forceinline__ void split2(float x, float y, unsigned (&part)[3]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  auto rounded = [](float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
  };
  auto low = [](unsigned two) { return __builtin_bit_cast(float, two << 16); };
  auto high = [](unsigned two) { return __builtin_bit_cast(float, two & 0xffff0000u); };
  part[0] = rounded(x, y);
  const float x1 = x - low(part[0]), y1 = y - high(part[0]);
  part[1] = rounded(x1, y1);
  const float x2 = x1 - low(part[1]), y2 = y1 - high(part[1]);
  part[2] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, y2), __builtin_bit_cast(unsigned, x2), 0x07060302u);
}
__device__ __forceinline__ void split(f32x4 v, u32x2 (&part)[3]) {
  unsigned low[3], high[3];
  split2(v[0], v[1], low);
  split2(v[2], v[3], high);
#pragma unroll
  for (int p = 0; p < 3; ++p) part[p] = u32x2{low[p], high[p]};
}

// Eight numbers' parts, as a lane's operands (with `negate` of their negatives).
__device__ __forceinline__ void parts(f32x4 low, f32x4 high, bool negate, bf16x8 (&out)[3]) {
  u32x2 p[3], q[3];
  split(negate ? -low : low, p);
  split(negate ? -high : high, q);
#pragma unroll
  for (int i = 0; i < 3; ++i) out[i] = __builtin_bit_cast(bf16x8, u32x4{p[i][0], p[i][1], q[i][0], q[i][1]});
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct SplitArgs {
  const float *a, *w;
  float* c;
  int M, N, K;
  int wide;                 // C's fours of columns begin on 16 bytes
  int tiles_m, tiles_n, panel;
};

// The elements (m, n) of the lanes in `bad`, made again (see above), one after the other: every lane
// of the wavefront takes part.
__device__ __noinline__ float made_again(float v, unsigned long long bad, const float* a, const float* b,
                                         int K, int m, int n) {
  const int lane = threadIdx.x % kWave;
  for (; bad; bad &= bad - 1) {
    const int of = __ffsll(bad) - 1;
    const float* x = a + (int64_t)__shfl(m, of, kWave) * K;
    const float* w = b + (int64_t)__shfl(n, of, kWave) * K;
    double sum = 0.;
    for (int k0 = 4 * lane; k0 - 4 * lane < K; k0 += 16 * kWave) {
      f32x4 xv[4], wv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + 4 * kWave * u;
        xv[u] = k < K ? *(const f32x4*)(x + k) : kZero, wv[u] = k < K ? *(const f32x4*)(w + k) : kZero;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum = fma((double)xv[u][j], (double)wv[u][j], sum);
      if (__any(sum != sum)) break;         // and it stays so
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
    if (lane == of) v = (float)sum;
  }
  return v;
}

// Stores a lane's four columns [n, n + 4) of row m; all lanes of a wavefront come here.
__device__ __forceinline__ void store4(const SplitArgs& a, f32x4 v, int m, int n) {
  const bool row = m < a.M;
  const bool fine = !row || fabsf(v[0]) + fabsf(v[1]) + fabsf(v[2]) + fabsf(v[3]) < INFINITY;
  if (__ballot(!fine)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned long long bad = __ballot(row && n + r < a.N && !(fabsf(v[r]) < INFINITY));
      if (bad) v[r] = made_again(v[r], bad, a.a, a.w, a.K, m, n + r);
    }
  }
  if (!row) return;
  float* out = a.c + (int64_t)m * a.N + n;
  if (n + 4 <= a.N && a.wide) {
    *(f32x4*)out = v;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) out[r] = v[r];
  }
}

// ---------------------------------------------------------------- few rows
// Up to 16 MT rows (48): a workgroup takes 16 columns, each of its eight wavefronts a run of K, so a
// weight is read once, a stretch ahead of its use.  Bound by the weights' way from memory.
template <int MT>
__global__ __launch_bounds__(kRuns* kWave) void gemm_f32_split_rows_kernel(SplitArgs a) {
  __shared__ __align__(16) float sums[kRuns][MT][256];
  const int run = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int l = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * 16;
  const int per = (a.K / 64 + kRuns - 1) / kRuns * 64, begin = run * per, end = min(begin + per, a.K);
  const float* w_row = a.w + (int64_t)min(n0 + l, a.N - 1) * a.K + 8 * g;
  const float* a_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = a.a + (int64_t)min(16 * i + l, a.M - 1) * a.K + 8 * g;
  f32x4 sum[MT], w[2][4], x[2][MT][4];      // [set][2 step + half]
#pragma unroll
  for (int i = 0; i < MT; ++i) sum[i] = kZero;
  auto fetch = [&](int set, int k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = k + u / 2 * 32 + u % 2 * 4;
      w[set][u] = *(const f32x4*)(w_row + at);
#pragma unroll
      for (int i = 0; i < MT; ++i) x[set][i][u] = *(const f32x4*)(a_row[i] + at);
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int step = 0; step < 2; ++step) {
      bf16x8 wp[3], xp[MT][3];
      f32x4 chain[MT];
      parts(w[set][2 * step], w[set][2 * step + 1], step & 1, wp);
#pragma unroll
      for (int i = 0; i < MT; ++i) parts(x[set][i][2 * step], x[set][i][2 * step + 1], false, xp[i]);
#pragma unroll
      for (int t = 0; t < kSmall; ++t)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          chain[i] = mfma(wp[kPartW[t]], xp[i][kPartA[t]], t ? chain[i] : kZero);
#pragma unroll
      for (int i = 0; i < MT; ++i) chain[i] += mfma(wp[0], xp[i][0], kZero);
#pragma unroll
      for (int i = 0; i < MT; ++i) sum[i] = step & 1 ? sum[i] - chain[i] : sum[i] + chain[i];
    }
  };
  if (begin < end) {
    fetch(0, begin);
    for (int k = begin; k < end; k += 128) {
      if (k + 64 < end) fetch(1, k + 64);
      multiply(0);
      if (k + 64 >= end) break;
      if (k + 128 < end) fetch(0, k + 128);
      multiply(1);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) *(f32x4*)&sums[run][i][lane * 4] = sum[i];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * 256; e += kRuns * kWave) {
    const int i = e / 256, row = e % 256 / 16, col = e % 16;
    const int at = (col / 4 * 16 + row) * 4 + col % 4;
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < kRuns; r += 2) v += sums[r][i][at] + sums[r + 1][i][at];
    // (whole wavefronts come here)
    const int m = 16 * i + row, n = n0 + col;
    const bool in = m < a.M && n < a.N;
    const unsigned long long bad = __ballot(in && !(fabsf(v) < INFINITY));
    if (bad) v = made_again(v, bad, a.a, a.w, a.K, m, n);
    if (in) a.c[(int64_t)m * a.N + n] = v;
  }
}

// ---------------------------------------------------------------- a run a wavefront
// A workgroup takes 16 TM rows and 16 TN columns (32 x 16 to 64 x 64), each of its eight wavefronts a run of K: what a
// wavefront cuts it multiplies itself, so nothing passes through LDS and nobody waits for others
// until the runs are added up.  Operands are sent for SETS steps of 32 ahead, into the registers
// that a step has just cut.
template <int TM, int TN, int SETS>      // SETS: 1 or 2
__global__ __launch_bounds__(kRuns* kWave) void gemm_f32_split_kernel(SplitArgs a) {
  constexpr int AT_ONCE = TN >= 4 ? 1 : TM;      // blocks of rows whose products go side by side
  extern __shared__ __align__(16) float sums[];  // [run][TM][TN][lane][4]
  const int run = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int l = lane % 16, g = lane / 16;

  // each XCD an eighth of the tiles, walked in panels (gemm_tiled_kernel.h); one row of tiles, whose
  // weights nobody shares, in the order of memory
  const int per_xcd = gridDim.x >> 3;
  const int tile = a.tiles_m > 1 ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
  if (tile >= a.tiles_m * a.tiles_n) return;
  const int panel = tile / (a.panel * a.tiles_n), in_panel = tile - panel * a.panel * a.tiles_n;
  const int height = min(a.panel, a.tiles_m - panel * a.panel);
  const int m0 = (panel * a.panel + in_panel % height) * 16 * TM, n0 = in_panel / height * 16 * TN;

  const int per = (a.K / 64 + kRuns - 1) / kRuns * 64;     // (the last runs may be shorter or empty)
  const int begin = run * per, end = min(begin + per, a.K);
  const float *w_row[TN], *a_row[TM];
#pragma unroll
  for (int j = 0; j < TN; ++j) w_row[j] = a.w + (int64_t)min(n0 + 16 * j + l, a.N - 1) * a.K + 8 * g;
#pragma unroll
  for (int i = 0; i < TM; ++i) a_row[i] = a.a + (int64_t)min(m0 + 16 * i + l, a.M - 1) * a.K + 8 * g;
  f32x4 sum[TM][TN], w[SETS][TN][2], x[SETS][TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = kZero;
  auto fetch = [](f32x4 (&to)[2], const float* from) {
    to[0] = *(const f32x4*)from;
    to[1] = *(const f32x4*)(from + 4);
  };
  if (begin < end) {
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      const int k = min(begin + 32 * s, end - 32);
#pragma unroll
      for (int j = 0; j < TN; ++j) fetch(w[s][j], w_row[j] + k);
#pragma unroll
      for (int i = 0; i < TM; ++i) fetch(x[s][i], a_row[i] + k);
    }
    for (int k0 = begin; k0 < end; k0 += 64) {
#pragma unroll
      for (int step = 0; step < 2; ++step) {
        const int s = step % SETS, ahead = min(k0 + 32 * (step + SETS), end - 32);
        bf16x8 wp[TN][3];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          parts(w[s][j][0], w[s][j][1], step & 1, wp[j]);
          fetch(w[s][j], w_row[j] + ahead);
        }
#pragma unroll
        for (int i0 = 0; i0 < TM; i0 += AT_ONCE) {
          bf16x8 xp[AT_ONCE][3];
          f32x4 chain[AT_ONCE][TN];
#pragma unroll
          for (int i = 0; i < AT_ONCE; ++i) {
            parts(x[s][i0 + i][0], x[s][i0 + i][1], false, xp[i]);
            fetch(x[s][i0 + i], a_row[i0 + i] + ahead);
          }
#pragma unroll
          for (int t = 0; t < kSmall; ++t)
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                chain[i][j] = mfma(wp[j][kPartW[t]], xp[i][kPartA[t]], t ? chain[i][j] : kZero);
#pragma unroll
          for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) chain[i][j] += mfma(wp[j][0], xp[i][0], kZero);
#pragma unroll
          for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              sum[i0 + i][j] = step & 1 ? sum[i0 + i][j] - chain[i][j] : sum[i0 + i][j] + chain[i][j];
        }
      }
    }
  }
  auto place = [&](int r, int block, int of) { return (f32x4*)(sums + ((r * TM * TN + block) * 64 + of) * 4); };
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) *place(run, i * TN + j, lane) = sum[i][j];
  __syncthreads();
  // a thread takes four columns of a row, a wavefront a block
  for (int e = threadIdx.x; e < TM * TN * 64; e += kRuns * kWave) {
    const int block = e / 64, of = e % 64;
    f32x4 v = kZero;
#pragma unroll
    for (int r = 0; r < kRuns; r += 2) v += *place(r, block, of) + *place(r + 1, block, of);
    store4(a, v, m0 + block / TN * 16 + of % 16, n0 + block % TN * 16 + of / 16 * 4);
  }
}

template <int TM, int TN, int SETS>
int launch_runs(SplitArgs a, hipStream_t stream) {
  auto* kernel = gemm_f32_split_kernel<TM, TN, SETS>;
  constexpr int lds = kRuns * TM * TN * 1024;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return -1;
  a.tiles_m = (a.M + 16 * TM - 1) / (16 * TM), a.tiles_n = (a.N + 16 * TN - 1) / (16 * TN);
  a.panel = a.tiles_m < 8 ? a.tiles_m : 8;
  const int per_xcd = (int)(((int64_t)a.tiles_m * a.tiles_n + 7) / 8);
  hipLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(kRuns * kWave), lds, stream, a);
  return 0;
}

// ---------------------------------------------------------------- tiles through LDS
// A BM x BN tile a workgroup, one a unit: G groups of GM x GN wavefronts, a group takes 8 / G runs
// of K.  A turn is 32 of K: operands come from memory into registers two turns ahead, are cut once
// for the whole group, between the products of the turn before, and put into the other of two LDS
// buffers.
// LDS: [part][row][32], a row's four pieces of 16 bytes at (piece ^ (row / 4 % 4)), so that the
// sixteen rows that a quarter of a wavefront reads fall into different banks.
template <int BM, int BN, int GM, int GN, int G>
__global__ __launch_bounds__(64 * GM * GN * G) void gemm_f32_split_tile_kernel(SplitArgs a) {
  constexpr int NW = GM * GN, THREADS = 64 * NW, TM = BM / GM / 16, TN = BN / GN / 16;
  constexpr int ROWS = BM + BN, PIECES = ROWS * 8, PER = (PIECES + THREADS - 1) / THREADS;
  constexpr int PART = ROWS * 64, BUFFER = 3 * PART, OWN = kRuns / G;
  static_assert(BM % (16 * GM) == 0 && BN % (16 * GN) == 0 && BM * 8 % THREADS == 0, "whole blocks");
  static_assert(G == 1 || OWN == 2, "a group's runs are one pair, or it has all of them");
  extern __shared__ __attribute__((aligned(16))) unsigned char split_lds[];
  const int lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave_all / NW, wave = wave_all % NW, wm = wave / GN, wn = wave % GN;

  // each XCD an eighth of the tiles, walked in panels (gemm_tiled_kernel.h)
  const int per_xcd = gridDim.x >> 3, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= a.tiles_m * a.tiles_n) return;
  const int panel = tile / (a.panel * a.tiles_n), in_panel = tile - panel * a.panel * a.tiles_n;
  const int height = min(a.panel, a.tiles_m - panel * a.panel);
  const int m0 = (panel * a.panel + in_panel % height) * BM, n0 = in_panel / height * BN;

  // turns of K: a group's runs (those behind K are empty), of one length for all groups; even
  const int run_turns = (a.K / 64 + kRuns - 1) / kRuns * 2, all_turns = a.K / 32;
  const int first = group * OWN * run_turns;
  const int turns = min(OWN * run_turns, all_turns);
  const int mine = max(min(turns, all_turns - first), 0);         // the others multiply nothing

  const float* from[PER];
  int to[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    // (pieces behind the tile's rows are the last row's again)
    const int piece = u * THREADS + wave * 64 + lane, row = min(piece / 8, ROWS - 1), c = piece % 8;
    from[u] = (row < BM ? a.a + (int64_t)min(m0 + row, a.M - 1) * a.K
                        : a.w + (int64_t)min(n0 + row - BM, a.N - 1) * a.K) + 4 * c;
    to[u] = row * 64 + ((c / 2) ^ (row / 4 % 4)) * 16 + c % 2 * 8;
  }
  unsigned char* buffers = split_lds + group * 2 * BUFFER;
  f32x4 next[2][PER];
  auto fetch_piece = [&](int set, int turn, int u) {
    const int64_t k = (int64_t)min(first + turn, all_turns - 1) * 32;
    next[set][u] = *(const f32x4*)(from[u] + k);
  };
  auto put_piece = [&](int set, int buffer, int u) {
    // (A's of every second turn)
    u32x2 part[3];
    split(buffer == 1 && u < BM * 8 / THREADS ? -next[set][u] : next[set][u], part);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(u32x2*)(buffers + buffer * BUFFER + p * PART + to[u]) = part[p];
  };
  const int at = l * 64 + ((g ^ (l / 4 % 4)) << 4);
  f32x4 run[TM][TN], pair[TM][TN], all[TM][TN];
  auto clear = [&](f32x4 (&sums)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[i][j] = kZero;
  };
  auto gather = [&](f32x4 (&sums)[TM][TN], const f32x4 (&more)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[i][j] += more[i][j];
  };
  auto turn = [&](int set, int t) {       // t even with set 0, odd with set 1
    const unsigned char* from_a = buffers + set * BUFFER + wm * TM * 1024 + at;
    const unsigned char* from_w = buffers + set * BUFFER + BM * 64 + wn * TN * 1024 + at;
    bf16x8 ap[3][TM], wp[3][TN];
    f32x4 step[TM][TN];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) ap[p][i] = *(const bf16x8*)(from_a + p * PART + i * 1024);
#pragma unroll
      for (int j = 0; j < TN; ++j) wp[p][j] = *(const bf16x8*)(from_w + p * PART + j * 1024);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next turn's pieces are cut between this one's products
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      put_piece(set ^ 1, set ^ 1, u);
      fetch_piece(set ^ 1, t + 3, u);
    }
#pragma unroll
    for (int term = 0; term < kSmall; ++term)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          step[i][j] = mfma(wp[kPartW[term]][j], ap[kPartA[term]][i], term ? step[i][j] : kZero);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) step[i][j] += mfma(wp[0][j], ap[0][i], kZero);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x4 more = G == 1 || t < mine ? step[i][j] : kZero;
        run[i][j] = set == 1 ? run[i][j] - more : run[i][j] + more;
      }
#pragma unroll
    for (int m = 0; m < kTerms * TM * TN; ++m) {
      __builtin_amdgcn_sched_group_barrier(8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(2, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // (loads stay on their way)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int u = 0; u < PER; ++u) fetch_piece(s, s, u);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    put_piece(0, 0, u);
    fetch_piece(0, 2, u);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  clear(all);
  int t = 0;
#pragma unroll 1
  for (int o = 0; o < OWN && t < turns; o += 2) {
    clear(pair);
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      clear(run);
      const int end = min((o + half + 1) * run_turns, turns);
#pragma unroll 1
      for (; t < end; t += 2) {
        turn(0, t);
        turn(1, t + 1);
      }
      gather(pair, run);
    }
    gather(all, pair);
  }
  if (G > 1) {
    // the other groups' pair of runs through LDS, [group - 1][wave][block][lane]
    auto place = [&](int gr, int i, int j) {
      return (f32x4*)(split_lds + (((((gr - 1) * NW + wave) * TM + i) * TN + j) * 64 + lane) * 16);
    };
    __syncthreads();
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *place(group, i, j) = all[i][j];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        for (int gr = 1; gr < G; ++gr) all[i][j] += *place(gr, i, j);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      store4(a, all[i][j], m0 + (wm * TM + i) * 16 + l, n0 + (wn * TN + j) * 16 + 4 * g);
}

template <int BM, int BN, int GM, int GN, int G>
int launch_tile(SplitArgs a, hipStream_t stream) {
  auto* kernel = gemm_f32_split_tile_kernel<BM, BN, GM, GN, G>;
  constexpr int lds = G * 2 * 3 * (BM + BN) * 64;
  static_assert(lds <= 160 * 1024 && (G - 1) * BM * BN * 4 <= lds, "LDS of a compute unit");
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return -1;
  a.tiles_m = (a.M + BM - 1) / BM, a.tiles_n = (a.N + BN - 1) / BN;
  a.panel = a.tiles_m < 8 ? a.tiles_m : 8;
  const int per_xcd = (int)(((int64_t)a.tiles_m * a.tiles_n + 7) / 8);
  hipLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(64 * GM * GN * G), lds, stream, a);
  return 0;
}

}  // namespace

int gemm_f32_split_launch(const float* A, const float* W, float* C, int M, int N, int K, int tile,
                          hipStream_t stream) {
  SplitArgs a{A, W, C, M, N, K, N % 4 == 0 && ((uintptr_t)C & 15) == 0, 0, 0, 1};
  const dim3 block(kRuns * kWave), grid((N + 15) / 16);
  if (tile == 0 && M <= 32) tile = M <= 16 ? 1 : 2;
  if (tile == 0) {
    // The tile with the least estimate: rounds of 256 units by what a tile takes, a part of its own
    // and one for every 1,024 of K, both measured with weights in memory.  (33 to 64 rows had a tile
    // of their own, 64 x 16, which reads all rows for every 16 columns: 4,096 x 4,096 53 to 56 us,
    // now 35 to 42, 1,024 x 3,072 32 to 36, now 21.)
    struct Tile { int bm, bn, most; float fixed_us, k_us; };
    constexpr Tile kTiles[] = {{48, 16, 48, 3.f, 8.f}, {32, 16, 0, 4.9f, 5.2f}, {32, 32, 0, 1.5f, 10.4f},
                               {32, 64, 0, 4.5f, 8.8f}, {64, 64, 0, 7.f, 14.f}, {128, 64, 0, 7.f, 30.f},
                               {128, 96, 0, 8.f, 41.f}, {128, 128, 0, 9.f, 49.5f}};
    float least = -1.f;
    for (int t = 0; t < 8; ++t) {
      if (kTiles[t].most && M > kTiles[t].most) continue;
      const int64_t tiles = (int64_t)((M + kTiles[t].bm - 1) / kTiles[t].bm) * ((N + kTiles[t].bn - 1) / kTiles[t].bn);
      const float us = (float)((tiles + 255) / 256) * (kTiles[t].fixed_us + kTiles[t].k_us * (float)K / 1024.f);
      if (least < 0.f || us < least) least = us, tile = t + 3;
    }
  }
  if (tile <= 3 && M > 16 * tile) return -1;
  switch (tile) {
    case 1: hipLaunchKernelGGL(gemm_f32_split_rows_kernel<1>, grid, block, 0, stream, a); return 0;
    case 2: hipLaunchKernelGGL(gemm_f32_split_rows_kernel<2>, grid, block, 0, stream, a); return 0;
    case 3: hipLaunchKernelGGL(gemm_f32_split_rows_kernel<3>, grid, block, 0, stream, a); return 0;
    case 4: return launch_runs<2, 1, 2>(a, stream);
    case 5: return launch_runs<2, 2, 2>(a, stream);
    case 6: return launch_tile<32, 64, 2, 2, 4>(a, stream);
    case 7: return launch_runs<4, 4, 1>(a, stream);
    case 8: return launch_tile<128, 64, 4, 2, 1>(a, stream);
    case 9: return launch_tile<128, 96, 4, 2, 1>(a, stream);
    case 10: return launch_tile<128, 128, 4, 2, 1>(a, stream);
    default: return -1;
  }
}

// The product by a tile's number (0: the sizes' choice), for tests and measuring; ts_gemm_fma is the
// call for everything else.
extern "C" int ts_gemm_f32_split(const float* a, const float* w, float* c, int M, int N, int K, int tile,
                                 hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || !gemm_f32_split_fits(K)) TS_FAIL("gemm_f32_split: K=%d is no multiple of 64", K);
  if (((uintptr_t)a | (uintptr_t)w) & 15) TS_FAIL("gemm_f32_split: operands must be 16-byte aligned");
  if (tile < 0 || tile > 10 || (tile >= 1 && tile <= 3 && M > 16 * tile))
    TS_FAIL("gemm_f32_split: tile %d does not take %d rows", tile, M);
  if (gemm_f32_split_launch(a, w, c, M, N, K, tile, stream))
    TS_FAIL("gemm_f32_split: a tile needs more LDS than the device gives");
  TS_CHECK_LAUNCH("gemm_f32_split");
  return 0;
}
