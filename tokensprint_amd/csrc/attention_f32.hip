// Paged causal attention of a float32 run on the float32 matrix cores: float32 queries and
// cache, head sizes of a multiple of 16 up to 128, up to 16 query heads a key/value head, pages
// of a multiple of 16 keys; what else there is goes to attention_generic.hip.
//
// A workgroup takes a tile of 16 rows (tokens of one entry x the query heads of a key/value head);
// its eight wavefronts take every eighth block of 64 keys, counted from position 0, and their
// results are merged in wavefront order.  So what a row adds up, and in which order, depends on
// its position and window alone, however the step was cut or batched.
//
// Scores are made transposed (keys x rows): a sum's registers then hold four consecutive keys of a
// row, which is what the product with the values takes as its operand, and that product, values
// transposed x weights, leaves four consecutive elements of a row in a register quadruple.  Nothing
// passes through LDS but the merge.  Keys and values come straight from their pages, 16 bytes a
// lane (values lie transposed in a page).
//
// What bounds it: at a prompt of 501 tokens (16 heads over 8, 128 wide) 1.1 GFLOP of useful
// products, 7 us at the float32 matrix rate, and a wavefront's chain of loads and products for
// each of its blocks.  The kernel before it, a workgroup per token and head with a key a lane,
// read every key row 32 times as 16-byte pieces 512 bytes apart.
#include "attention_mfma.h"
#include <type_traits>

int ts_check_attention_args(const AttentionArgs& a, const char* who);

namespace {

constexpr int kWaves = 8;
constexpr int kBlock = 64;                 // keys of a block

__device__ __forceinline__ f32x4 read4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}

// NT: sixteenths of the head size.  EXTRAS: scores are more than scale times the product.
template <int NT, bool EXTRAS>
__global__ __launch_bounds__(kWaves* kWave) void attention_f32_kernel(AttentionMfmaArgs m) {
  constexpr int HD = 16 * NT, LD = HD + 4;
  extern __shared__ __align__(16) float lds[];
  float* o_s = lds;                                   // [kWaves][16][LD]
  float* m_s = o_s + kWaves * 16 * LD;                // [kWaves][16]
  float* l_s = m_s + kWaves * 16;                     // [kWaves][16]
  const AttentionArgs& a = m.base;
  const int tile = blockIdx.x, kvh = blockIdx.y, group = m.rows_per_token;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int l = lane % 16, g = lane / 16, P = a.page_size;
  const int entry = m.tiles ? m.tiles[3 * tile] : tile;
  const int first = m.tiles ? m.tiles[3 * tile + 1] : a.q_start[tile];
  const int tokens = m.tiles ? m.tiles[3 * tile + 2] : 1;
  // column l of a score tile: query head l % group of the tile's token l / group
  const bool mine = l < tokens * group;
  const int token = first + (mine ? l / group : 0), head = kvh * group + (mine ? l % group : 0);
  const int pos = a.positions[token], from = first_visible(a, pos);
  const int last = a.positions[first + tokens - 1], begin = first_visible(a, a.positions[first]);
  const int* table = a.table + (int64_t)entry * a.table_width;
  const float* q = (const float*)a.q + ((int64_t)token * a.nq + head) * HD + 4 * g;
  ScoreExtra x;
  if (EXTRAS) x = score_extra(a, head, pos);
  f32x4 qf[NT], o[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) qf[j] = read4(q + 16 * j);
  float top, sum;                          // of column l; `sum` of this lane's keys only
  // The wavefront's blocks.  A key that a row does not see has no weight with it, but nothing times
  // a value that is not finite is not nothing: APART makes the product with the values once a
  // row, without the keys that the row does not see, and takes the row's column of it.
  auto walk = [&](auto apart) {
    constexpr bool APART = decltype(apart)::value;
#pragma unroll
    for (int j = 0; j < NT; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    top = -INFINITY, sum = 0.f;
    int b = begin / kBlock;
    b += (w - b) & (kWaves - 1);             // the first block of this wavefront's
    for (; b * kBlock <= last; b += kWaves) {
      // (every load is made, from page 0 where there is none: what it brings is not used)
      int64_t row[4];                        // of the block's four tiles of 16 keys: their page
      bool have[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int key = b * kBlock + 16 * t;
        const int page = __builtin_amdgcn_readfirstlane(table[min(key, last) / P]);
        have[t] = key <= last && page >= 0;
        row[t] = ((int64_t)max(page, 0) * a.nkv + kvh) * P * HD;
      }
      f32x4 kf[4][NT], vf[4][NT], s[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float* k = (const float*)a.k_pages + row[t] + (int64_t)((b * kBlock + 16 * t) % P + l) * HD + 4 * g;
#pragma unroll
        for (int j = 0; j < NT; ++j) kf[t][j] = read4(k + 16 * j);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NT; ++j) s[t] = mfma4(kf[t][j], qf[j], s[t]);
      }
      __builtin_amdgcn_sched_barrier(0);     // (the values in the keys' registers)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float* v = (const float*)a.v_pages + row[t] + (int64_t)l * P + (b * kBlock + 16 * t) % P + 4 * g;
#pragma unroll
        for (int c = 0; c < NT; ++c) vf[t][c] = read4(v + (int64_t)16 * c * P);
      }
      __builtin_amdgcn_sched_barrier(0);
      float high = top;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = b * kBlock + 16 * t + 4 * g + r;
          const float v = EXTRAS ? extra_score(x, s[t][r], key) : s[t][r] * a.scale;
          s[t][r] = have[t] && mine && key <= pos && key >= from ? v : -INFINITY;
          high = fmaxf(high, s[t][r]);
        }
      high = fmaxf(high, __shfl_xor(high, 16, kWave));
      high = fmaxf(high, __shfl_xor(high, 32, kWave));
      // (`high` stays -inf only while the row has seen no key: zeros are kept)
      const float fall = high == -INFINITY ? 1.f : expf(top - high);
      top = high;
      sum *= fall;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[t][r] = s[t][r] == -INFINITY ? 0.f : expf(s[t][r] - high);
          sum += s[t][r];
        }
#pragma unroll
      for (int c = 0; c < NT; ++c) o[c] *= fall;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int key = b * kBlock + 16 * t;
        if (!have[t] || key + 15 > last) {   // a page's places behind the last key hold anything
#pragma unroll
          for (int c = 0; c < NT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (!have[t] || key + 4 * g + r > last) vf[t][c][r] = 0.f;
        }
        if constexpr (APART) {
#pragma unroll 1
          for (int row = 0; row < tokens * group; ++row) {
            const int to = __shfl(pos, row, kWave), lo = __shfl(from, row, kWave);
#pragma unroll
            for (int c = 0; c < NT; ++c) {
              f32x4 sums = o[c];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const bool sees = key + 4 * g + r <= to && key + 4 * g + r >= lo;
                sums = __builtin_amdgcn_mfma_f32_16x16x4f32(sees ? vf[t][c][r] : 0.f, s[t][r], sums, 0, 0, 0);
              }
              if (l == row) o[c] = sums;
            }
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < NT; ++c)
              o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][c][r], s[t][r], o[c], 0, 0, 0);
        }
      }
    }
  };
  walk(std::false_type{});
  // (a value of that kind leaves NaN in every row that meets it, whatever comes behind)
  bool nan = false;
#pragma unroll
  for (int c = 0; c < NT; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) nan = nan || o[c][r] != o[c][r];
  if (__builtin_amdgcn_ballot_w64(nan && mine) != 0) walk(std::true_type{});
  sum += __shfl_xor(sum, 16, kWave);
  sum += __shfl_xor(sum, 32, kWave);
  if (g == 0) {
    m_s[w * 16 + l] = top;
    l_s[w * 16 + l] = sum;
  }
#pragma unroll
  for (int c = 0; c < NT; ++c)
    *reinterpret_cast<f32x4*>(o_s + (w * 16 + l) * LD + 16 * c + 4 * g) = o[c];
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * HD / 4; i += kWaves * kWave) {
    const int r = i / (HD / 4), d = i % (HD / 4) * 4;
    if (r >= tokens * group) break;
    float all = -INFINITY, den = 0.f;
#pragma unroll
    for (int u = 0; u < kWaves; ++u) all = fmaxf(all, m_s[u * 16 + r]);
    f32x4 num = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
      const float mu = m_s[u * 16 + r];
      if (mu == -INFINITY) continue;       // a wavefront without keys
      const float weight = expf(mu - all);
      if (weight == 0.f) continue;         // (its sums may be infinite)
      den += l_s[u * 16 + r] * weight;
      num += read4(o_s + (u * 16 + r) * LD + d) * weight;
    }
    const int h = kvh * group + r % group;
    if (a.sink) den += expf(fminf(a.sink[h] - all, 69.f));
    *reinterpret_cast<f32x4*>((float*)a.out + ((int64_t)(first + r / group) * a.nq + h) * HD + d) =
        num * (den > 0.f ? 1.f / den : 0.f);
  }
}

template <int NT>
int launch(const AttentionMfmaArgs& m, hipStream_t stream) {
  const size_t lds = sizeof(float) * kWaves * 16 * (16 * NT + 4 + 2);
  const bool extras = has_score_extras(m.base);
  const void* fn = extras ? (const void*)attention_f32_kernel<NT, true> : (const void*)attention_f32_kernel<NT, false>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return -1;
  const dim3 grid(m.num_tiles, m.base.nkv), block(kWaves * kWave);
  if (extras) hipLaunchKernelGGL((attention_f32_kernel<NT, true>), grid, block, lds, stream, m);
  else hipLaunchKernelGGL((attention_f32_kernel<NT, false>), grid, block, lds, stream, m);
  return 0;
}

}  // namespace

// Whether this kernel takes float32 attention of these sizes.
extern "C" int ts_attention_f32_fits(int hd, int group, int page_size, int nkv, int keep) {
  return hd > 0 && hd % 16 == 0 && hd <= 128 && group >= 1 && group <= 16 && page_size > 0 &&
         page_size % 16 == 0 && nkv <= 65535 && keep == 0;
}

// `args`: base, tiles (or null: a token an entry), num_tiles, rows_per_token (the query heads of a
// key/value head); a tile holds up to 16 / rows_per_token tokens.
extern "C" int ts_attention_f32(const AttentionMfmaArgs* args, hipStream_t stream) {
  const AttentionMfmaArgs& m = *args;
  const AttentionArgs& a = m.base;
  if (a.num_tokens <= 0 || m.num_tiles <= 0) return 0;
  if (ts_check_attention_args(a, "attention_f32")) return -1;
  if (!ts_attention_f32_fits(a.hd, a.nq / a.nkv, a.page_size, a.nkv, a.keep) ||
      m.rows_per_token != a.nq / a.nkv ||
      (((uintptr_t)a.q | (uintptr_t)a.out | (uintptr_t)a.k_pages | (uintptr_t)a.v_pages) & 15))
    TS_FAIL("attention_f32: hd=%d nq=%d nkv=%d page_size=%d keep=%d", a.hd, a.nq, a.nkv, a.page_size, a.keep);
  int rc;
  switch (a.hd / 16) {
    case 1: rc = launch<1>(m, stream); break;
    case 2: rc = launch<2>(m, stream); break;
    case 3: rc = launch<3>(m, stream); break;
    case 4: rc = launch<4>(m, stream); break;
    case 5: rc = launch<5>(m, stream); break;
    case 6: rc = launch<6>(m, stream); break;
    case 7: rc = launch<7>(m, stream); break;
    default: rc = launch<8>(m, stream); break;
  }
  if (rc != 0) TS_FAIL("attention_f32: hd=%d needs more LDS than the device gives", a.hd);
  TS_CHECK_LAUNCH("attention_f32");
  return 0;
}
