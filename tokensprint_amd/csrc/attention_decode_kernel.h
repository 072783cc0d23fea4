// The kernel of attention_decode.hip as a template, so that its forms with and without
// score extras compile in translation units of their own, side by side.
#pragma once
#include <type_traits>
#include "attention_core.h"

struct AttentionDecodeArgs {
  AttentionMfmaArgs m;      // tiles = null, num_tiles = entries = tokens
  const bf16_t* qkv;        // fused: [T, (nq + 2 * kv_in_row) * hd + row_extra]; else null
  const float* q_weight;    // [hd] or null: no norm
  const float* k_weight;
  const float* cos;         // [max_pos, hd / 2] or null: no rotation
  const float* sin;
  float eps;
  int kv_in_row;            // nkv: the row brings k and v, written to the cache here; 0: q only
  int defer_merge;          // 1: with more than one split, leave the partial results unmerged
                            // (ts_gemm_tail_merged_bf16 or ts_attention_merge takes them)
  unsigned* arrivals;       // [items] zeros, or null.  Given (and the merge not deferred), the
                            // workgroup of an item that finishes last merges the splits itself
                            // and leaves the item's count at zero: no merge kernel
  int row_extra;            // further columns of a qkv row behind the heads
};

int launch_attention_merge(const AttentionMfmaArgs& args, hipStream_t stream);

template <int HD> constexpr int decode_waves() { return HD <= 128 ? 8 : 4; }
// floats of a row of partial sums in LDS: neighbouring rows start four banks apart
template <int HD> constexpr int merge_row() { return HD + 4; }

// What the host works out for the kernel: the divisions by numbers that are the same for all.
struct DecodeShape {
  unsigned group;                  // query heads of a key/value head
  unsigned heads, heads_inv;       // workgroups of an entry (key/value heads times blocks of their heads)
  unsigned splits_inv;
};

// A lane's share of a head vector while it is normed and turned: four elements of the first half and
// the four that they turn with.  HD / 8 lanes hold a head, so a wavefront does several at once (four
// of 128 elements) and nothing crosses lanes but the sum of squares.  One wavefront does this while
// the others wait for it, so what counts is how many instructions it issues (1.8 ns each) and how
// many loads stand before its last: in the operand's layout, a quarter of a head to a lane and most
// lanes without a row, this was 0.8 us of a step's 7.5 at one request.
template <int HD>
struct HeadShare {
  static constexpr int USED = HD / 8;                                           // lanes of a head
  static constexpr int LANES = USED <= 4 ? 4 : USED <= 8 ? 8 : USED <= 16 ? 16 : 32;
  static constexpr int AT_ONCE = kWave / LANES;
  bf16x4 lo, hi;
  __device__ __forceinline__ void load(const bf16_t* head, int c) {
    lo = *(const bf16x4*)(head + c * 4);
    hi = *(const bf16x4*)(head + HD / 2 + c * 4);
  }
  // where element e (a multiple of 4) of operand row `row` of `rows` stands, in units of four
  static __device__ __forceinline__ int place(int e, int row, int rows) {
    return ((e % (HD / 4) / 8 * 4 + e / (HD / 4)) * rows + row) * 2 + e % 8 / 4;
  }
  __device__ __forceinline__ void store(bf16x4* operand, int c, int row, int rows) const {
    operand[place(c * 4, row, rows)] = lo;
    operand[place(HD / 2 + c * 4, row, rows)] = hi;
  }
  __device__ __forceinline__ void prepare(bool norm, const f32x4 (&w)[2], float eps, bool turn, const f32x4& cs,
                                          const f32x4& sn, int c) {
    float x[4], y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { x[j] = (float)lo[j]; y[j] = (float)hi[j]; }
    if (norm) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) ss = fmaf(y[j], y[j], fmaf(x[j], x[j], ss));
      if (USED < LANES && c >= USED) ss = 0.f;
      // the neighbour's, the other pair's, then mirrored eights and sixteens
      auto add_from = [&](auto lanes) {
        ss += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), decltype(lanes)::value, 0xf, 0xf, true));
      };
      add_from(std::integral_constant<int, 0xB1>());
      add_from(std::integral_constant<int, 0x4E>());
      if (LANES >= 8) add_from(std::integral_constant<int, 0x141>());
      if (LANES >= 16) add_from(std::integral_constant<int, 0x140>());
      if (LANES >= 32) {
        auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(ss), __float_as_uint(ss), false, false);
        ss = __uint_as_float(a[0]) + __uint_as_float(a[1]);
      }
      const float rstd = rsqrtf(ss / (float)HD + eps);
#pragma unroll
      for (int j = 0; j < 4; ++j) { x[j] *= rstd * w[0][j]; y[j] *= rstd * w[1][j]; }
    }
    if (turn) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = x[j], b = y[j];
        x[j] = a * cs[j] - b * sn[j];
        y[j] = b * cs[j] + a * sn[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) { lo[j] = (bf16_t)x[j]; hi[j] = (bf16_t)y[j]; }
  }
};

// A float32 to memory, and back, at device scope without ordering: such accesses pass the
// caches that another XCD does not share.
__device__ __forceinline__ void store_past_caches(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_past_caches(float* p, float v, float w) {     // p: of 8 bytes
  __hip_atomic_store((uint64_t*)p, (uint64_t)__float_as_uint(w) << 32 | __float_as_uint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_past_caches(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The merge of attention_merge_kernel (same order, same arithmetic per element, so the same
// bits) by the THREADS threads of one workgroup, over the `used` first splits of one item:
// slot (first_slot + split * 16 + row) holds a row's statistics and HD partial sums.  A
// thread takes E elements and asks for all of a group of GROUP splits of each before it uses the first:
// the workgroup's last act, bound by its trips to memory and by its instructions (two elements a
// thread and always eight splits: 1.5 us of 10.9 for four splits of 2 rows of 128, with one and four 0.8;
// more splits and more than an element to a thread, two at a time: 16 query heads of 128 over one key/value head,
// 2,000 tokens, 15.4 us one at a time, 14.5).
template <int HD, int THREADS, int GROUP, int E>
__device__ __forceinline__ void merge_splits_here(const float* partial_o, const float* partial_ml,
                                                  int64_t first_slot, int used, int rows, bf16_t* out,
                                                  const float* sink = nullptr, int first_head = 0) {
  partial_o += first_slot * HD;
  partial_ml += first_slot * 2;
  const int count = rows * HD;
  for (int e0 = threadIdx.x; e0 < count; e0 += E * THREADS) {
    int row[E], d[E];
    float M[E], L[E], acc[E];
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int e = E == 1 ? e0 : min(e0 + k * THREADS, count - 1);    // past the end: the last again, not stored
      row[k] = e / HD;
      d[k] = e % HD;
      M[k] = -INFINITY;
      L[k] = acc[k] = 0.f;
    }
    for (int s0 = 0; s0 < used; s0 += GROUP) {
      float ms[E][GROUP], ls[E][GROUP], part[E][GROUP];
#pragma unroll
      for (int j = 0; j < GROUP; ++j)
#pragma unroll
        for (int k = 0; k < E; ++k) {
          const unsigned slot = min(s0 + j, used - 1) * 16 + row[k];
          const uint64_t ml = __hip_atomic_load((const uint64_t*)partial_ml + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ms[k][j] = __uint_as_float((unsigned)ml);
          ls[k][j] = __uint_as_float((unsigned)(ml >> 32));
          part[k][j] = load_past_caches(partial_o + slot * HD + d[k]);
        }
#pragma unroll
      for (int k = 0; k < E; ++k) {
        float Mg = M[k];
#pragma unroll
        for (int j = 0; j < GROUP; ++j) Mg = (s0 + j < used) ? fmaxf(Mg, ms[k][j]) : Mg;
        if (Mg == -INFINITY) continue;
        const float keep = __builtin_amdgcn_exp2f(M[k] - Mg);
        L[k] *= keep;
        acc[k] *= keep;
#pragma unroll
        for (int j = 0; j < GROUP; ++j) {
          const bool live = s0 + j < used && ms[k][j] != -INFINITY;
          const float w = live ? __builtin_amdgcn_exp2f(ms[k][j] - Mg) : 0.f;
          L[k] += live ? ls[k][j] * w : 0.f;
          acc[k] += live ? part[k][j] * w : 0.f;
        }
        M[k] = Mg;
      }
    }
#pragma unroll
    for (int k = 0; k < E; ++k) {
      if (E > 1 && e0 + k * THREADS >= count) break;
      const float sum = sum_with_sink(L[k], M[k], sink, first_head + row[k]);
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      out[(int64_t)row[k] * HD + d[k]] = (bf16_t)(acc[k] * inv);
    }
  }
}

// The entry with the rank-th longest context of up to 64 (equal ones in order), and its position.
struct Ranked {
  int entry, pos;
};
__device__ __forceinline__ Ranked ranked_entry(const int* positions, int entries, int rank, int lane) {
  const int pos = positions[min(lane, entries - 1)];
  const int key = lane < entries ? pos * 64 + 63 - lane : -1;
  int before = 0;
#pragma unroll
  for (int j = 0; j < kWave; ++j) before += __builtin_amdgcn_readlane(key, j) > key ? 1 : 0;
  const int entry = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lane < entries && before == rank));
  return {entry, __builtin_amdgcn_readlane(pos, entry)};
}

// EXTRA: scores with a cap, a distance bias or a query temperature (attention.h).
// RANKED (more items than the chip has units, up to 64 entries, no splits): the items are the entries'
// in the order of their contexts, longest first.  A unit holds one workgroup at a time (its eight
// wavefronts take over 200 registers), so a long context that comes late is walked alone at the end: 64
// entries of 100 to 2,047 tokens in no order 64.3 us (4.4 TB/s), ranked 55.9 (5.0), of 128 to 4,096
// tokens 117.9 and 99.4 (5.6), 40 entries 50.7 and 41.7; entries of one length, which have nothing to
// rank, 54.4 and 55.6.  A captured step's contexts are known on the device only, so every wavefront
// ranks them for itself.  (Workgroups of four wavefronts, two to a unit: 61.1 and 114 us, ranked too.)
template <int HD, bool FUSED, bool EXTRA, bool RANKED = false>
__global__ __launch_bounds__(decode_waves<HD>() * kWave) void attention_decode_kernel(
    AttentionDecodeArgs args, DecodeShape sh) {
  constexpr int NW = decode_waves<HD>();
  constexpr int DB = HD / 16, KS = (HD + 31) / 32;
  const AttentionMfmaArgs& ma = args.m;
  const AttentionArgs& a = ma.base;
  const int wave = uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int group = sh.group;
  const int item = blockIdx.x, split = blockIdx.y;
  // a division by a number the compiler does not know costs 40 instructions before the first load
  Ranked place{(int)divided(item, sh.heads, sh.heads_inv), 0};
  int kvh = item - place.entry * sh.heads, hb = 0;
  if (ma.head_blocks > 1) { hb = kvh % ma.head_blocks; kvh /= ma.head_blocks; }
  if constexpr (RANKED) place = ranked_entry(a.positions, ma.num_tiles, place.entry, lane);
  const int entry = place.entry;
  const int token = entry;
  const int* table = a.table + (int64_t)entry * a.table_width;

  const int hh = hb * 16 + r;                                 // head inside the group
  const bool row_ok = r < ma.rows_per_token && hh < group;
  const int head = kvh * group + min(hh, group - 1);
  // Fused form: the last wave does not walk; it prepares the query rows for the others.
  // In the first split the wave before it does not walk either: it takes the new key,
  // side by side with the last wave's work on the queries.  What those two need from
  // memory is asked for first of all, before anything else is worked out: the head
  // vector and the norm weight at once, cos and sin as soon as the position is here.
  const bool new_key = FUSED && args.kv_in_row > 0;           // the step's own key is not in the cache yet
  const bool adds_new = new_key && split == 0;                // this workgroup brings the new key in
  const bool prep_wave = FUSED && wave == NW - 1;
  const bool key_wave = adds_new && wave == NW - 2;
  const bool walker = !prep_wave && !key_wave;
  const int pos_lane = RANKED ? place.pos : a.positions[token];
  const int rows = min(ma.rows_per_token, group - hb * 16);
  using Share = HeadShare<HD>;
  const int share_row = lane / Share::LANES, share_lane = lane % Share::LANES;
  const int share_at = min(share_lane, Share::USED - 1);
  const bf16_t* row = FUSED ? args.qkv : nullptr;
  if (FUSED) row += (int64_t)token * ((a.nq + 2 * args.kv_in_row) * HD + args.row_extra);
  Share part;
  f32x4 pw[2], cs, sn;
  bf16x4 nv[DB], nv_slot = {0, 0, 0, 0};       // the new key's value: as a partial sum, and as its slot takes it
  const float* prep_weight = nullptr;
  const bf16_t* first_head = nullptr;          // of the query heads, or the new key
  if constexpr (FUSED) {
    if (!walker) {
      prep_weight = prep_wave ? args.q_weight : args.k_weight;
      first_head = row + (int64_t)(prep_wave ? kvh * group + hb * 16 : a.nq + kvh) * HD;
      part.load(first_head + (int64_t)(prep_wave ? min(share_row, rows - 1) : 0) * HD, share_at);
      if (prep_weight) {
        pw[0] = *(const f32x4*)(prep_weight + share_at * 4);
        pw[1] = *(const f32x4*)(prep_weight + HD / 2 + share_at * 4);
      }
    }
  }
  const int pos = uniform(pos_lane);
  if constexpr (FUSED) {
    if (!walker) {
      if (args.cos != nullptr) {
        cs = *(const f32x4*)(args.cos + (int64_t)pos * (HD / 2) + share_at * 4);
        sn = *(const f32x4*)(args.sin + (int64_t)pos * (HD / 2) + share_at * 4);
      }
      if (key_wave) {
        const bf16_t* vrow = row + (int64_t)(a.nq + args.kv_in_row + kvh) * HD;
#pragma unroll
        for (int db = 0; db < DB; ++db) nv[db] = *(const bf16x4*)(vrow + db * 16 + g * 4);
        nv_slot = *(const bf16x4*)(vrow + min(r, DB - 1) * 16 + g * 4);
      }
    }
  }
  int new_page = -1;
  if (FUSED && key_wave && hb == 0 && pos >= 0) new_page = ((ConstTable)table)[pos >> __builtin_ctz(a.page_size)];
  const int last = new_key ? pos - 1 : pos;                   // last key walked from the cache
  const int lo = first_visible(a, pos);
  // chunks of this split: the arithmetic of attention_merge (from pos, not from last)
  const KeyWalk walk = key_walk<32>(a, lo);
  const int c_first = walk.origin / kChunk, c_last = pos / kChunk;
  const int per = divided(c_last - c_first + ma.num_splits, ma.num_splits, sh.splits_inv);
  const int c0 = c_first + split * per, c1 = min(c0 + per, c_last + 1);
  if (c0 > c_last) {   // more splits than chunks: a neutral partial, no data touched
    if (g == 0 && wave == 0) {
      const int64_t slot = ((int64_t)item * ma.num_splits + split) * 16 + r;
      ma.partial_ml[slot * 2] = -INFINITY;
      ma.partial_ml[slot * 2 + 1] = 0.f;
    }
    return;
  }

  const int walkers = FUSED ? NW - 1 - (adds_new ? 1 : 0) : NW;

  TileState<HD> t;
  t.pos = row_ok ? last : -1;
  t.lo = lo;
  t.keep = a.keep;
  const float scale_log2 = a.scale * 1.44269504088896341f;
  ScoreExtraLog2 x;
  if (EXTRA) x = in_log2(score_extra(a, head, row_ok ? pos : -1));   // distances from the query's own position
  const int stride = walkers * 32;
  const int key_begin = max(c0 * kChunk, walk.origin) + wave * 32;
  const int key_end = (prep_wave || key_wave) ? 0 : min(c1 * kChunk, last + 1);
  PageCursor cur{(ConstTable)table, a.page_size, last, walk, -1, -1};
  KvBlock<HD> A, B;
  // Head sizes in whole 32-element slices take the blocks with 16-byte value loads.  Ranked items are
  // more than the chip has units and wait for memory, not for a unit's loads: their keys go straight
  // into the operand's order (64 entries of 100 to 2,047 tokens, whole steps: 2,472 us spread through
  // LDS, 2,457 straight; of 128 to 4,096 tokens at the 8B shape 1,193 and 1,172).  Above 128 it is the
  // registers of two blocks that count, and what is left for the compiler to send loads ahead with: us
  // straight / through LDS, 40 entries of 2,500 tokens, ranked (8 key/value heads) 160 113 / 98, 192 123 / 117, 224
  // 143 / 138, 256 173 / 161; 20 entries of 8 heads or 40 of 4, not ranked, 160 56 / 61, 192 84 / 81, 224 112 / 113,
  // 256, one request of 800, 25 / 23.
  constexpr bool kWide = HD % 32 == 0, kStraight = RANKED ? HD <= 128 : HD == 160 || HD == 224;
  auto load_block = [&](KvBlock<HD>& b, int kb) {
    if constexpr (kWide && kStraight) load_kv_block_wide<HD>(b, a, cur, kvh, kb, stride, r, g);
    else if constexpr (kWide) load_kv_block_rows<HD>(b, a, cur, kvh, kb, stride, lane);
    else load_kv_block<HD, true>(b, a, table, cur, kvh, kb, stride, r, g);
  };

  if constexpr (FUSED) {
    // The last wave prepares the query rows for all of them (through LDS): the others
    // have their first key block in flight meanwhile.
    __shared__ bf16x8 s_q[KS * kWave];         // [slice][lane of the operand]
    __shared__ bf16x8 s_k[KS * 4];             // the new key: [slice][g]
    const bool rotate = args.cos != nullptr;
    if (walker) {
      cur.start(key_begin);
      if (key_begin < key_end) load_block(A, key_begin);
    }
    if (!walker) {
      if (prep_wave) {
        for (int row0 = 0;;) {
          Share coming = part;
          if (row0 + Share::AT_ONCE < rows)
            coming.load(first_head + (int64_t)min(row0 + Share::AT_ONCE + share_row, rows - 1) * HD, share_at);
          part.prepare(prep_weight != nullptr, pw, args.eps, rotate, cs, sn, share_lane);
          if (share_lane < Share::USED && row0 + share_row < rows)
            part.store((bf16x4*)s_q, share_lane, row0 + share_row, 16);
          row0 += Share::AT_ONCE;
          if (row0 >= rows) break;
          part = coming;
        }
      } else {
        part.prepare(prep_weight != nullptr, pw, args.eps, rotate, cs, sn, share_lane);
        if (lane < Share::USED) part.store((bf16x4*)s_k, lane, 0, 1);
      }
    }
    __syncthreads();
    const int q_row = g * 16 + min(r, rows - 1);      // rows past the last take its query: nobody reads them
#pragma unroll
    for (int s = 0; s < KS; ++s) t.q[s] = s_q[s * kWave + q_row];
#pragma unroll
    for (int db = 0; db < DB; ++db) t.o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    t.m = -INFINITY;
    t.l = 0.f;

    if (key_wave) {
      f32x4 dots = {0.f, 0.f, 0.f, 0.f};                    // every row of the product's keys is the new key
#pragma unroll
      for (int s = 0; s < KS; ++s)
        dots = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s_k[s * 4 + g], t.q[s], dots, 0, 0, 0);
      const float dot = dots[0];
      // this wave's partial: one key with weight 1
      t.m = EXTRA ? extra_score_log2(x, dot, pos)
                  : dot * scale_log2;
      t.l = g == 0 ? 1.f : 0.f;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x4 v = nv[db];
        t.o[db] = f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
      }
    }
  } else {
    cur.start(key_begin);
    if (key_begin < key_end) load_block(A, key_begin);
    load_query<HD>(t, (const bf16_t*)a.q + ((int64_t)token * a.nq + head) * HD, row_ok, g);
  }

  extern __shared__ __attribute__((aligned(16))) unsigned char merge_lds[];
  // a wavefront's keys are spread where its partial sums will stand: nobody else's
  unsigned char* scratch = merge_lds + NW * kWave * 2 * 4 + wave * (16 * merge_row<HD>() * 4);
  auto update = [&](KvBlock<HD>& b, int v) {
    if constexpr (kWide && !kStraight) spread_keys<HD>(b, scratch, lane);
    const int kb = walk.real(v);
    tile_update<HD, false, kWide, EXTRA>(t, b, kb, scale_log2, kb + 31 <= last && kb >= lo, g, &x);
  };
  for (int v = key_begin; v < key_end; v += 2 * stride) {
    if (v + stride < key_end)
      load_block(B, v + stride);
    update(A, v);
    if (v + stride >= key_end) break;
    if (v + 2 * stride < key_end)
      load_block(A, v + 2 * stride);
    update(B, v + stride);
  }
  f32x4 (&o)[DB] = t.o;
  float m = t.m, l = row_sum<HD>(t);

  // The waves' partial results (the new key's among them) all go to LDS, and every wave
  // merges, in wave order, its share of the head's blocks of 16 elements and stores that
  // share: the merge is as wide as the workgroup instead of one wave's long tail.
  float (*s_ml)[kWave][2] = (float (*)[kWave][2])merge_lds;                        // [NW]
  constexpr int kRow = merge_row<HD>();
  float (*s_o)[16][kRow] = (float (*)[16][kRow])(merge_lds + NW * kWave * 2 * 4);    // [NW]
  s_ml[wave][lane][0] = m;
  s_ml[wave][lane][1] = l;
#pragma unroll
  for (int db = 0; db < DB; ++db) *(f32x4*)&s_o[wave][r][db * 16 + g * 4] = o[db];
  __syncthreads();
  if constexpr (FUSED) {
    // The new key and value into the cache slot of position pos, once per key/value head: behind
    // the last barrier that others wait at, with nothing loaded after them here (loads and stores
    // share a counter, and a wait for a load would wait for these).
    if (key_wave && hb == 0) {
      const int P = a.page_size, off = pos & (P - 1);
      if (new_page >= 0) {
        bf16_t* kdst = (bf16_t*)a.k_pages + (((int64_t)new_page * a.nkv + kvh) * P + off) * HD;
        if (lane < Share::USED) {
          *(bf16x4*)(kdst + lane * 4) = part.lo;
          *(bf16x4*)(kdst + HD / 2 + lane * 4) = part.hi;
        }
        bf16_t* vdst = (bf16_t*)a.v_pages + ((int64_t)new_page * a.nkv + kvh) * HD * P + off;
        if (r < DB) {
#pragma unroll
          for (int i = 0; i < 4; ++i) vdst[(int64_t)(r * 16 + g * 4 + i) * P] = nv_slot[i];
        }
      }
    }
  }
  constexpr int kShare = (DB + NW - 1) / NW;         // blocks of 16 elements per wave
  // Merge by the last to finish: the partial results go out past the caches (their readers
  // may sit on another XCD, behind another L2), each wave waits until its own have been
  // taken, the workgroup counts itself in at the item's counter, and the one that finds
  // all the others there reads every split's result back the same way and merges them in
  // the order and arithmetic of attention_merge.  Nothing here needs the caches written
  // back or dropped, which is what release and acquire at device scope would cost.
  const bool fold = ma.num_splits > 1 && !args.defer_merge && args.arrivals != nullptr;
  const bool has_share = rows * HD <= NW * kWave ? wave * kWave < rows * HD : wave * kShare < DB;
  if (!has_share && !fold) return;
  const int64_t slot = ((int64_t)item * ma.num_splits + split) * 16 + r;
  if (rows * HD <= NW * kWave) {
    // few rows (4 of 128): an element a thread, which is a quarter of the instructions that the
    // operand's layout takes with most of its rows empty (0.3 us of 5.6)
    const int e = threadIdx.x, mrow = e / HD, d = e % HD;
    if (mrow < rows) {
      float mw[NW], lw[NW], ow[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) { mw[w] = s_ml[w][mrow][0]; lw[w] = s_ml[w][mrow][1]; ow[w] = s_o[w][mrow][d]; }
      float M = mw[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) M = fmaxf(M, mw[w]);
      const float Mc = M == -INFINITY ? 0.f : M;      // (no key: all weights are 0)
      float acc = 0.f, sum = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float ww = __builtin_amdgcn_exp2f(mw[w] - Mc);
        sum = fmaf(lw[w], ww, sum);
        acc += ww == 0.f ? 0.f : ow[w] * ww;
      }
      const int h = kvh * group + hb * 16 + mrow;
      if (ma.num_splits == 1) {
        sum = sum_with_sink(sum, M, a.sink, h);
        const float inv = sum > 0.f ? 1.f / sum : 0.f;
        ((bf16_t*)a.out)[((int64_t)token * a.nq + h) * HD + d] = (bf16_t)(acc * inv);
      } else {
        const int64_t at_slot = ((int64_t)item * ma.num_splits + split) * 16 + mrow;
        float* po = ma.partial_o + at_slot * HD + d;
        float* pm = ma.partial_ml + at_slot * 2;
        if (fold) {
          store_past_caches(po, acc);
          if (d == 0) store_past_caches(pm, M, sum);
        } else {
          *po = acc;
          if (d == 0) { pm[0] = M; pm[1] = sum; }
        }
      }
    }
  } else if (has_share) {
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, s_ml[w][lane][0]);
    float ww[NW];
    l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = s_ml[w][lane][0];
      // a wave that saw no key has m = -inf (and so has everyone if M is): weight 0
      ww[w] = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
      l += s_ml[w][lane][1] * ww[w];
    }
    m = M;
    // lane (r, g) holds O^T[d = db*16 + g*4 + i][row r]
    // the sink joins the sum where the row is finished: here only without key splits
    const float whole = ma.num_splits == 1 ? sum_with_sink(l, m, a.sink, head) : l;
    const float inv = whole > 0.f ? 1.f / whole : 0.f;
#pragma unroll
    for (int k = 0; k < kShare; ++k) {
      const int db = wave * kShare + k;
      if (db >= DB) break;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const f32x4 ow = *(const f32x4*)&s_o[w][r][db * 16 + g * 4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += ww[w] == 0.f ? 0.f : ow[i] * ww[w];   // never 0 * garbage
      }
      if (!row_ok) continue;
      if (ma.num_splits == 1) {
        bf16x4 ov = {(bf16_t)(acc[0] * inv), (bf16_t)(acc[1] * inv), (bf16_t)(acc[2] * inv),
                     (bf16_t)(acc[3] * inv)};
        *(bf16x4*)((bf16_t*)a.out + ((int64_t)token * a.nq + head) * HD + db * 16 + g * 4) = ov;
      } else if (fold) {
#pragma unroll
        for (int i = 0; i < 4; ++i) store_past_caches(ma.partial_o + slot * HD + db * 16 + g * 4 + i, acc[i]);
      } else {
        *(f32x4*)(ma.partial_o + slot * HD + db * 16 + g * 4) = acc;
      }
    }
    if (ma.num_splits > 1 && wave == 0 && g == 0) {
      if (fold) {
        store_past_caches(ma.partial_ml + slot * 2, m, l);
      } else {
        ma.partial_ml[slot * 2] = m;
        ma.partial_ml[slot * 2 + 1] = l;
      }
    }
  }
  if (!fold) return;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);                     // this wave's stores have been taken
  __shared__ unsigned s_before;
  __syncthreads();
  if (threadIdx.x == 0)
    s_before = __hip_atomic_fetch_add(args.arrivals + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  // splits that hold chunks: the arithmetic of attention_merge; the others have returned
  const int nchunks = c_last - c_first + 1;
  const int used = min(ma.num_splits, (nchunks + per - 1) / per);
  if ((int)s_before + 1 != used) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (threadIdx.x == 0)
    __hip_atomic_store(args.arrivals + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  bf16_t* out = (bf16_t*)a.out + ((int64_t)token * a.nq + kvh * group + hb * 16) * HD;
  auto merge = [&](auto at_once, auto each) {
    merge_splits_here<HD, NW * kWave, decltype(at_once)::value, decltype(each)::value>(
        ma.partial_o, ma.partial_ml, (int64_t)item * ma.num_splits * 16, used, rows, out, a.sink, kvh * group + hb * 16);
  };
  constexpr std::integral_constant<int, 1> one;
  constexpr std::integral_constant<int, 2> two;
  constexpr std::integral_constant<int, 4> four;
  constexpr std::integral_constant<int, 8> eight;
  // (up to four splits an element at a time whatever a thread has: four at a time 8.1 us in place of 7.0 where it
  // has two, and a fourth form beside these three costs every launch 0.15)
  if (__builtin_expect(used <= 4, 1)) merge(four, one);
  else if (__builtin_expect(rows * HD <= NW * kWave, 1)) merge(eight, one);
  else merge(eight, two);
}

int launch_attention_merge(const AttentionMfmaArgs& args, hipStream_t stream);

template <int HD, bool EXTRA, bool RANKED = false>
static int launch_decode(const AttentionDecodeArgs& args, hipStream_t stream) {
  const AttentionMfmaArgs& m = args.m;
  const int items = m.num_tiles * m.base.nkv * m.head_blocks;
  const AttentionArgs& a = m.base;
  const unsigned heads = a.nkv * m.head_blocks;
  const DecodeShape sh{(unsigned)(a.nq / a.nkv), heads, inverse32(heads), inverse32(m.num_splits)};
  const dim3 grid(items, m.num_splits), block(decode_waves<HD>() * kWave);
  // the merge area: per wave its row statistics and HD/16 blocks of partial sums
  const size_t lds = (size_t)decode_waves<HD>() * (kWave * 2 * 4 + 16 * merge_row<HD>() * 4);
  if (args.qkv) {
    if constexpr (HD % 32 == 0) {
      auto kernel = attention_decode_kernel<HD, true, EXTRA, RANKED>;
      static bool raised = false;     // per head size
      if (lds > 48 * 1024 && !raised) {
        if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess)
          TS_FAIL("attention_decode: cannot raise the LDS limit to %zu bytes", lds);
        raised = true;
      }
      hipLaunchKernelGGL(kernel, grid, block, lds, stream, args, sh);
    } else {
      TS_FAIL("attention_decode: the fused form needs a head size that is a multiple of 32");
    }
  } else {
    auto kernel = attention_decode_kernel<HD, false, EXTRA>;
    static bool raised = false;
    if (lds > 48 * 1024 && !raised) {
      if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds) != hipSuccess)
        TS_FAIL("attention_decode: cannot raise the LDS limit to %zu bytes", lds);
      raised = true;
    }
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, args, sh);
  }
  if (m.num_splits > 1 && !args.defer_merge && !args.arrivals) return launch_attention_merge(m, stream);
  return 0;
}

