// Paged causal attention of long portions of prompts, 32 query rows a wavefront (bfloat16,
// head sizes 64 and 128, pages of a power of two from 16 up), as a template so that its forms
// compile in translation units of their own.
//
// What bounds it: at 8,192 tokens of 64 query heads, where it takes 1,043 us (1,050 TFLOP/s; with 16 rows
// a wavefront 1,394), the card's power (before sums were rescaled for every new largest score, zeros in
// place of ordinary data took 812 instead of 1,005); at 2,048 tokens of 16 (36 us, before 40) the longest
// item, and 8 us of launch and dependent trips to memory.  Thirty-two rows
// a wavefront halve what LDS has to read out per product and the softmax's instructions; a row's
// scores lie in two lanes, so its maximum is one exchange.  The scores of the next block and the values
// of the one before beside a block's softmax, in one wavefront, was slower (all 256 registers; 1,106 us).
#pragma once
#include "attention_core.h"

typedef __attribute__((ext_vector_type(16))) float f32x16;

// 64 x 16 bytes from a uniform base and the lanes' byte offsets to LDS at `lds` + 16 * lane,
// without registers in between.  (Written as an instruction: the compiler, knowing that such a
// load writes LDS, makes LDS reads wait for every one of them in flight.  The kernel counts
// these loads itself and separates them from the reads by a barrier.)
__device__ __forceinline__ void lds_dma16_at(const char* base, unsigned offset, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(offset), "s"(base), "s"(lds)
               : "memory", "m0");
}

// The larger of the two values that lanes l and l + 32 hold, in both; their sum.
__device__ __forceinline__ float halves_max(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return max2(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Layouts (v_mfma_f32_32x32x16_bf16, lane = 32 * h + c):
//   K operand    lane (c, h) holds K[key sigma(c)][16 s + 8 h + j]                 (A of S^T = K Q^T)
//   Q operand    lane (c, h) holds Q[row c][16 s + 8 h + j]                        (B)
//   S^T result   register i of lane (c, h): key sigma(8 (i / 4) + 4 h + i % 4), query row c
//   V operand    lane (c, h) holds V^T[32 db + c][keys 8 h .. 8 h + 7 of a page's sixteen]
//   O^T result   register i of lane (c, h): element 32 db + 8 (i / 4) + 4 h + i % 4, query row c
// sigma exchanges bits 2 and 3 of a key's number, so that registers 8 t .. 8 t + 7 of a lane are
// keys 16 t + 8 h .. + 7 and, rounded, its part of the second product's operand where they are.
//
// TILES wavefronts share an item's key blocks (an item is 2 TILES consecutive 16-row tiles), KEYS
// keys a turn; SETS such sets split the item's turns (set s takes turns s, s + SETS, ...), each with a
// ring of two buffers, and merge through LDS at the end.
template <int HD, int TILES, int SETS, int KEYS, bool P16, bool EXTRA>
__device__ __forceinline__ void attention_prefill_tall(const AttentionMfmaArgs& args) {
  constexpr int KS = HD / 16, DB = HD / 32, B = KEYS / 32, G = KEYS / 16;
  constexpr int SUB = HD / 32;                 // slots of 1 KB per sixteen keys
  constexpr int L = G * SUB / TILES;           // of a turn's keys, that a wavefront sends for
  constexpr int OFFS = SUB > TILES ? SUB / TILES : 1;
  constexpr int VALUES = KEYS * HD * 2;        // bytes of a turn's keys; its values lie behind them
  constexpr int BUF = 2 * VALUES;
  static_assert((HD == 64 || HD == 128) && G * SUB % TILES == 0, "rows of 128 or 256 bytes, whole slots");
  extern __shared__ __attribute__((aligned(1024))) unsigned char prefill_lds[];
  const AttentionArgs& a = args.base;
  const int wave_all = uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int wave = wave_all % TILES, set = SETS == 1 ? 0 : wave_all / TILES;
  const int c = lane % 32, h = lane / 32;
  const int group = a.nq / a.nkv;
  const int heads = a.nkv * args.head_blocks;
  const int head_slot = blockIdx.x % heads;                   // one head per XCD's L2
  const int rank = blockIdx.x / heads;
  const int kvh = head_slot / args.head_blocks;
  const int hb = head_slot % args.head_blocks;
  const int P = a.page_size, lp = __builtin_ctz(P);
  const int tq = 16 / args.rows_per_token;                    // tokens of sixteen rows
  float scale_log2 = a.scale * 1.44269504088896341f;

  // Where things lie in LDS.  A key's row, in key order, its 16-byte pieces exchanged so that
  // the sixteen rows that lanes read together lie in different banks; values as their pages hold
  // them (a head element's sixteen keys, 32 bytes), halves exchanged every eight elements for
  // the same reason.  Neighbouring lanes then name neighbouring pieces: a compute unit takes a load of
  // 1 KB in 18 cycles where they do, in 66 where each names 16 bytes in a line that its neighbours do not (in
  // the order of the operands, 32 lines in all).
  unsigned k_off[OFFS], v_off[OFFS];           // of this lane's piece in its sixteen keys, bytes
#pragma unroll
  for (int i = 0; i < OFFS; ++i) {
    constexpr int ROWS = 1024 / (HD * 2), PIECES = HD / 8;      // keys of a slot, pieces of a key
    const int sub = (wave + TILES * i) % SUB;
    const int key = sub * ROWS + lane / PIECES;
    const int f = HD == 128 ? key : key / 2 % 8;
    k_off[i] = 2u * (key * HD + (((lane % PIECES) ^ f) * 8));
    v_off[i] = 2u * ((sub * 32 + lane / 2) * P + (((lane % 2) ^ (lane / 16 % 2)) * 8));
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)prefill_lds + set * 2 * BUF;
  const unsigned char* ring = prefill_lds + set * 2 * BUF;
  const int key_c = (c & 0x13) | ((c & 4) << 1) | ((c & 8) >> 1);       // sigma(c)
  const int key_f = HD == 128 ? key_c % 16 : key_c % 16 / 2;
  const unsigned k_read = key_c * (HD * 2), k_piece = h ^ key_f;
  const unsigned v_read = VALUES + (2 * c + (h ^ (c / 8 % 2))) * 16;

  const char* k_head = (const char*)a.k_pages + (int64_t)kvh * P * HD * 2;
  const char* v_head = (const char*)a.v_pages + (int64_t)kvh * HD * P * 2;
  const int64_t page_stride = 2 * (int64_t)a.nkv * P * HD;    // bytes, keys and values alike

  // the item, and the lane's row of it
  const int entry = uniform(args.tiles[rank * 3]), tok0 = uniform(args.tiles[rank * 3 + 1]),
            ntok = uniform(args.tiles[rank * 3 + 2]);
  const int in16 = c % 16 / args.rows_per_token;
  const int ti = (wave * 2 + c / 16) * tq + in16;
  const int hh = hb * 16 + c % 16 % args.rows_per_token;
  const int head = kvh * group + min(hh, group - 1);
  const bool row_ok = in16 < tq && ti < ntok && hh < group;
  bf16x8 q[KS];
  {
    const bf16_t* qrow = (const bf16_t*)a.q + ((int64_t)(tok0 + min(ti, ntok - 1)) * a.nq + head) * HD;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < KS; ++s) q[s] = row_ok ? *(const bf16x8*)(qrow + 16 * s + 8 * h) : zero8;
  }
  const int pos_first = uniform(a.positions[tok0]);           // positions are consecutive
  const ConstTable table = (ConstTable)(a.table + (int64_t)entry * a.table_width);
  const int pos_last = pos_first + ntok - 1;
  const int lo_all = first_visible(a, pos_first);

  const int row_pos = row_ok ? pos_first + ti : -1;
  const int row_lo = first_visible(a, row_pos);
  ScoreExtraLog2 x;
  if (EXTRA) x = in_log2(score_extra(a, head, row_pos));
  // the wavefront's tokens (scalars)
  const int t0 = wave * 2 * tq, t1 = min(ntok, (wave + 1) * 2 * tq);
  const int tile_first = pos_first + t0;
  const int tile_last = t0 < ntok ? pos_first + t1 - 1 : -1;
  const int tile_lo = first_visible(a, tile_first);
  const int tile_lo_last = first_visible(a, tile_last);

  // The item's turns, numbered from its first; this set takes turns set, set + SETS, ...:
  // `mine` of them, numbered j here.  Every set passes the same number of barriers.
  const KeyWalk walk = key_walk<KEYS>(a, lo_all);
  const int key_begin = walk.origin;
  const int nturns = (pos_last - key_begin) / KEYS + 1;
  const int rounds = (nturns + SETS - 1) / SETS;
  const int mine = (nturns - set + SETS - 1) / SETS;
  const int kb_first = key_begin + KEYS * set;
  const int last_page = pos_last >> lp;              // the last page the item may name
  // page ids of the turn that will be sent for next (a page beyond the item's last is the last
  // again, one that a window has let go reads page 0: their keys are masked, and what the cache
  // holds is finite)
  int nx[G];
  typedef int Ids __attribute__((ext_vector_type(G), aligned(4)));
  auto fetch_ids = [&](int v) {
    const int kb = walk.real(v);
    const int i0 = kb >> lp;
    if (P16 && i0 + G - 1 <= last_page) {        // consecutive pages: one scalar load
      const Ids ids = *(const Ids __attribute__((address_space(4)))*)(table + i0);
#pragma unroll
      for (int g = 0; g < G; ++g) nx[g] = ids[g];
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g) nx[g] = table[min((kb + 16 * g) >> lp, last_page)];
    }
  };
  fetch_ids(kb_first);
  auto issue = [&](int j, int to) {
    const int v = kb_first + KEYS * SETS * j, kb = walk.real(v);
#pragma unroll
    for (int i = 0; i < L; ++i) {
      // slot wave + TILES i of the turn's: sixteen keys number slot / SUB
      int g, id;
      if constexpr (SUB >= TILES) {
        g = TILES * i / SUB;
        id = nx[g];
      } else {
        g = wave / SUB + TILES / SUB * i;
        id = nx[TILES / SUB * i];
#pragma unroll
        for (int n = 1; n < TILES / SUB; ++n) id = wave / SUB == n ? nx[TILES / SUB * i + n] : id;
      }
      const int64_t page = max(id, 0) * page_stride;
      const int in = P16 ? 0 : (kb + 16 * g) & (P - 1);
      const unsigned dst = lds0 + to * BUF + (wave + TILES * i) * 1024;
      lds_dma16_at(k_head + page + in * (HD * 2), k_off[i % OFFS], dst);
      lds_dma16_at(v_head + page + in * 2, v_off[i % OFFS], dst + VALUES);
    }
    fetch_ids(v + KEYS * SETS);
  };

  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m = -INFINITY, l = 0.f;      // l: this lane's share of the row's sum

  auto work = [&](int kb, const unsigned char* buf) {
    // a step's operands are asked for ahead of its products
    constexpr int AHEAD = 8 / B < KS ? 8 / B : KS;
    bf16x8 kf[AHEAD][B];
    auto read_keys = [&](int s) {
      const unsigned char* at = buf + k_read + ((k_piece ^ (2 * s)) * 16);
#pragma unroll
      for (int b = 0; b < B; ++b) kf[s % AHEAD][b] = *(const bf16x8*)(at + b * (32 * HD * 2));
    };
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) read_keys(s);
    f32x16 st[B];
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) st[b][i] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int b = 0; b < B; ++b)
        st[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s % AHEAD][b], q[s], st[b], 0, 0, 0);
      if (s + AHEAD < KS) read_keys(s + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
    bf16x8 vf[G][DB];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int db = 0; db < DB; ++db) vf[g][db] = *(const bf16x8*)(buf + v_read + (g * SUB + db) * 1024);
    __builtin_amdgcn_sched_barrier(0);
    const int at = kb + 8 * h;       // register i of block b: key at + 32 b + 16 (i / 8) + i % 8
    if (EXTRA) {
      if (x.capped) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[b][i] = capped_log2(x, st[b][i]);
      } else {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[b][i] *= x.row;
      }
      if (x.sloped) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[b][i] = off_by_distance(x, st[b][i], at + 32 * b + 16 * (i / 8) + i % 8);
      }
      scale_log2 = 1.f;
    }
    if (!(kb + KEYS - 1 <= tile_first && kb >= tile_lo_last)) {
      asm volatile("" ::: "memory");   // keeps this a branch
      // (a key's number is a constant beyond the lane's first: the row's bounds are brought
      // there once a turn, so no register holds a key's)
      const int last = row_pos - at, lowest = row_lo - at, kept = a.keep - at;
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int n = 32 * b + 16 * (i / 8) + i % 8;
          st[b][i] = (n <= last && (n >= lowest || n < kept)) ? st[b][i] : -INFINITY;
        }
    }
    float mx[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      mx[b] = st[b][0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx[b] = max2(mx[b], st[b][i]);
    }
    // The weights are relative to the row's largest score so far, and what has been summed is rescaled
    // for rows that have met a larger one.  (A reference left up to 2^8 below it, as published attention
    // kernels have it, saves most of that, 1,015 us in place of 1,043 at 8,192 tokens of 64 heads, but a row's
    // largest weight is then no longer the one that bfloat16 holds exactly: rows that few keys dominate
    // were 1.14 to 1.25 times as far from float64.  A condition of the lane's, not of the wavefront's: the sums
    // then stay in the registers they are in, where the compiler would copy all 64 beside a branch that the
    // wavefront takes as one; without a condition 18.5 in place of 18.8 us at 1,024 tokens of 16, 1,072 at the
    // 8,192 of 64.)
    const float top = halves_max(B == 2 ? max2(mx[0], mx[B - 1]) : mx[0]) * scale_log2;
    if (top > m) {
      const float corr = __builtin_amdgcn_exp2f(m - max2(top, -1e30f));
      m = top;
      l *= corr;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= corr;
    }
    const float m_use = max2(m, -1e30f);
    bf16x8 pv[G];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(st[b][i], scale_log2, -m_use));
        ps += p;
        pv[2 * b + i / 8][i % 8] = (bf16_t)p;
      }
      l += ps;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[g][db], pv[g], o[db], 0, 0, 0);
  };

  // the query rows are waited for once, not at their first use inside the loop, where the wait
  // would be for every load in flight as well
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(q[s]));
  __builtin_amdgcn_s_waitcnt(0x0F70);
  if (mine > 0) issue(0, 0);
  for (int j = 0; j < rounds; ++j) {
    const int kb = walk.real(kb_first + KEYS * SETS * j);
    __builtin_amdgcn_s_waitcnt(0x0F70);        // this wavefront's share of turn j has arrived
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();              // everyone's has, and everyone is through with turn j - 1
    asm volatile("" ::: "memory");
    if (j + 1 < mine) issue(j + 1, (j + 1) & 1);
    if (j < mine && kb <= tile_last && (kb + KEYS - 1 >= tile_lo || kb < a.keep)) work(kb, ring + (j & 1) * BUF);
  }

  l = halves_sum(l);                           // (by all lanes: it crosses lanes)
  bf16_t* out = (bf16_t*)a.out + ((int64_t)(tok0 + ti) * a.nq + head) * HD;
  // Unit u of the results: registers 8 (u % 2) .. + 7 of o[u / 2], elements 16 u + 4 h .. + 3 and
  // 16 u + 8 + 4 h .. + 3.  The lane's halves exchange four each, and a lane has eight in a row.
  auto store_unit = [&](int u, const float* v) {
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    typedef unsigned U4 __attribute__((ext_vector_type(4)));
    bf16x4 lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = (bf16_t)v[i], hi[i] = (bf16_t)v[4 + i];
    const U2 y = __builtin_bit_cast(U2, lo), z = __builtin_bit_cast(U2, hi);
    auto s0 = __builtin_amdgcn_permlane32_swap(y[0], z[0], false, false);
    auto s1 = __builtin_amdgcn_permlane32_swap(y[1], z[1], false, false);
    const U4 eight = {s0[0], s1[0], s0[1], s1[1]};
    if (row_ok) *(U4*)(out + 16 * u + 8 * h) = eight;
  };
  if constexpr (SETS == 1) {
    const float sum = sum_with_sink(l, m, a.sink, head);
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
    for (int u = 0; u < 2 * DB; ++u) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = o[u / 2][8 * (u % 2) + i] * inv;
      store_unit(u, v);
    }
  } else {
    // The sets leave their results in LDS, in the rings' space: [set][tile][register][lane], the
    // row statistics behind them; each then adds up its share of the units, set by set.
    constexpr int REGS = DB * 16, UNITS = 2 * DB / SETS;
    static_assert(2 * DB % SETS == 0, "whole units");
    float* lds_o = (float*)prefill_lds;
    float* lds_ml = lds_o + SETS * TILES * REGS * kWave;
    __syncthreads();                             // the rings have been read for the last time
#pragma unroll
    for (int i = 0; i < REGS; ++i) lds_o[(wave_all * REGS + i) * kWave + lane] = o[i / 16][i % 16];
    lds_ml[wave_all * 2 * kWave + lane] = m;
    lds_ml[(wave_all * 2 + 1) * kWave + lane] = l;
    __syncthreads();
    float ms[SETS], w[SETS], m_use = -1e30f, sum = 0.f;
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      ms[s] = lds_ml[(s * TILES + wave) * 2 * kWave + lane];
      m_use = max2(m_use, ms[s]);
    }
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      // (a set that saw no key of this row has m = -inf and weight 0)
      w[s] = __builtin_amdgcn_exp2f(ms[s] - m_use);
      sum += lds_ml[((s * TILES + wave) * 2 + 1) * kWave + lane] * w[s];
    }
    sum = sum_with_sink(sum, m_use, a.sink, head);
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
    for (int n = 0; n < UNITS; ++n) {
      const int u = set * UNITS + n;
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int s = 0; s < SETS; ++s) v[i] += lds_o[((s * TILES + wave) * REGS + u * 8 + i) * kWave + lane] * w[s];
        v[i] *= inv;
      }
      store_unit(u, v);
    }
  }
}

// Two wavefronts a SIMD in every form: two workgroups of one set of four beside rings of 64 KB (head
// size 128), or one of eight wavefronts.
template <int HD, int TILES, int SETS, int KEYS, bool P16, bool EXTRA>
__global__ __launch_bounds__(kWave * TILES * SETS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attention_prefill_tall_kernel(AttentionMfmaArgs args) {
  attention_prefill_tall<HD, TILES, SETS, KEYS, P16, EXTRA>(args);
}

template <int HD, int TILES, int SETS, int KEYS, bool EXTRA>
int launch_prefill_tall(const AttentionMfmaArgs& args, hipStream_t stream) {
  const int heads = args.base.nkv * args.head_blocks;
  constexpr int rings = SETS * 2 * KEYS * HD * 4, merge = SETS == 1 ? 0 : SETS * TILES * (HD / 2 + 2) * kWave * 4;
  constexpr int lds = rings > merge ? rings : merge;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  const bool p16 = args.base.page_size == 16;
  void (*kernel)(AttentionMfmaArgs) = p16 ? attention_prefill_tall_kernel<HD, TILES, SETS, KEYS, true, EXTRA>
                                               : attention_prefill_tall_kernel<HD, TILES, SETS, KEYS, false, EXTRA>;
  static bool raised[2] = {false, false};     // per instantiation
  if (!raised[p16]) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      TS_FAIL("attention_prefill: cannot raise the LDS limit to %d bytes", lds);
    raised[p16] = true;
  }
  hipLaunchKernelGGL(kernel, dim3(args.num_tiles * heads), dim3(kWave * TILES * SETS), lds, stream, args);
  return 0;
}
