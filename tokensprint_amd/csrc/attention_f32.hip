// Paged causal attention of a float32 run on the float32 matrix cores: float32 queries and
// cache, head sizes of a multiple of 16 up to 128, up to 16 query heads a key/value head, pages
// of a multiple of 16 keys; what else there is goes to attention_generic.hip.
//
// A workgroup takes a tile of 16 rows (tokens of one entry x the query heads of a key/value head);
// its eight wavefronts take every eighth block of 16 keys, counted from position 0, and their
// results are merged in wavefront order.  So what a row adds up, and in which order, depends on
// its position and window alone, however the step was cut or batched.
//
// Scores are made transposed (keys x rows): a sum's registers then hold four consecutive keys of a
// row, which is what the product with the values takes as its operand, and that product, values
// transposed x weights, leaves four consecutive elements of a row in a register quadruple.  Nothing
// passes through LDS but the merge.  Keys and values come straight from their pages, 16 bytes a
// lane (values lie transposed in a page).
//
// A wavefront asks for a block's values before its scores and for the next block's keys behind them,
// in the registers of the keys that the scores have used: 16 loads are under way beneath each of its
// two products.  Blocks of 64 keys, all loaded and then waited for, left half of the wavefronts of a
// prompt of 501 tokens without a block.  Blocks of 32 in this form spill.
//
// The tiles of all heads lie one behind the other in the grid, heads fastest: the longest tiles of every
// head begin first, and with eight heads an XCD has one head's pages in its cache.
//
// What bounds it: at a prompt of 501 tokens (16 heads over 8, 128 wide) 1.1 GFLOP of useful products, 7 us
// at the float32 matrix rate, and two wavefronts a SIMD (registers) whose products wait for the scores'
// maximum and their loads.  Measured, blocks of 64 -> here: 501 tokens 43.5 -> 29.6 us, 2,048 tokens
// 305 -> 245, 32 heads 68.5 -> 54.8, 64 single tokens over 100 to 1,990 positions 148 -> 112, one over
// 501 21.4 -> 18.5.  Error against float64 (relative, 501 tokens): 3.1e-7 -> 2.0e-7; two chains of
// products make a score.
#include "attention_mfma.h"
#include <type_traits>

int ts_check_attention_args(const AttentionArgs& a, const char* who);

namespace {

constexpr int kWaves = 8;
constexpr int kBlock = 16;                 // keys of a block
constexpr int kGridTiles = 32768;          // tiles in the grid's second dimension

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
  const int tile = blockIdx.z * kGridTiles + blockIdx.y, kvh = blockIdx.x, group = m.rows_per_token;
  if (tile >= m.num_tiles) return;
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
    f32x4 kf[NT], vf[NT], s;
    int page;                                // of the block whose keys are loaded or under way
    bool have;                               // whether the block that has scores has a page
    // (every load is made, from page 0 where there is none: what it brings is not used)
    auto place = [&] { return ((int64_t)max(page, 0) * a.nkv + kvh) * P * HD; };
    auto load_keys = [&](int b) {            // b * kBlock <= last
      page = __builtin_amdgcn_readfirstlane(table[b * kBlock / P]);
      const float* k = (const float*)a.k_pages + place() + (int64_t)(b * kBlock % P + l) * HD + 4 * g;
#pragma unroll
      for (int j = 0; j < NT; ++j) kf[j] = read4(k + 16 * j);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto score = [&](int b) {
      have = page >= 0;
      const float* v = (const float*)a.v_pages + place() + (int64_t)l * P + b * kBlock % P + 4 * g;
#pragma unroll
      for (int c = 0; c < NT; ++c) vf[c] = read4(v + (int64_t)16 * c * P);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 chain[2] = {};
#pragma unroll
      for (int j = 0; j < NT; ++j) chain[j & 1] = mfma4(kf[j], qf[j], chain[j & 1]);
      s = chain[0] + chain[1];
      __builtin_amdgcn_sched_barrier(0);     // (the next keys in these keys' registers)
    };
    auto add = [&](int b) {
      const int key = b * kBlock + 4 * g;    // of s[0]
      float high = top;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = EXTRAS ? extra_score(x, s[r], key + r) : s[r] * a.scale;
        s[r] = have && mine && key + r <= pos && key + r >= from ? v : -INFINITY;
        high = fmaxf(high, s[r]);
      }
      high = fmaxf(high, __shfl_xor(high, 16, kWave));
      high = fmaxf(high, __shfl_xor(high, 32, kWave));
      // (`high` stays -inf only while the row has seen no key: zeros are kept)
      const float fall = high == -INFINITY ? 1.f : expf(top - high);
      top = high;
      sum *= fall;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[r] = s[r] == -INFINITY ? 0.f : expf(s[r] - high);
        sum += s[r];
      }
#pragma unroll
      for (int c = 0; c < NT; ++c) o[c] *= fall;
      // (a page's places behind the last key hold anything; selects: as a branch for the last block
      // alone it became a branch for each register of every block)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool there = have && key + r <= last;
#pragma unroll
        for (int c = 0; c < NT; ++c) vf[c][r] = there ? vf[c][r] : 0.f;
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
              const bool sees = key + r <= to && key + r >= lo;
              sums = __builtin_amdgcn_mfma_f32_16x16x4f32(sees ? vf[c][r] : 0.f, s[r], sums, 0, 0, 0);
            }
            if (l == row) o[c] = sums;
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int c = 0; c < NT; ++c)
            o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[c][r], s[r], o[c], 0, 0, 0);
      }
    };
    int b = begin / kBlock;
    b += (w - b) & (kWaves - 1);             // the first block of this wavefront's
    if (b * kBlock > last) return;
    load_keys(b);
#pragma unroll 1
    for (; (b + kWaves) * kBlock <= last; b += kWaves) {
      score(b);
      load_keys(b + kWaves);
      add(b);
    }
    score(b);
    add(b);
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
  const dim3 grid(m.base.nkv, min(m.num_tiles, kGridTiles), (m.num_tiles + kGridTiles - 1) / kGridTiles);
  const dim3 block(kWaves * kWave);
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
