// Paged causal attention on the matrix cores for long portions of prompts (bfloat16).
//
// The tile list comes sorted by the length of the key range, longest first.
//
// A wavefront works on TPW consecutive 16-row query tiles of one batch entry and walks
// their common key range alone, 32 keys at a time, with the next block's keys and values
// in flight while the current block is worked on.  Every K and V block it loads serves
// TPW tiles; the four waves of a workgroup take neighbouring tiles, so most of their
// loads meet in the first-level cache.  A tile skips blocks beyond its causal range or
// before its window, and skips the mask where every key of a block is visible.
#include "attention_core.h"

#include <algorithm>
#include <cmath>
#include <exception>
#include <vector>

template <int HD, int TPW, bool PAGE16>
__global__ __launch_bounds__(256) void attention_prefill_kernel(AttentionMfmaArgs args) {
  const AttentionArgs& a = args.base;
  const int wave = uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int group = a.nq / a.nkv;
  // Workgroups are handed to the eight XCDs in turn, and each XCD has an L2 of its own:
  // workgroup b works on head (b mod heads), so a head's keys and values stay in one L2.
  // Its four waves take neighbouring query tiles, the longest key ranges first.
  const int heads = a.nkv * args.head_blocks;
  const int head_slot = blockIdx.x % heads;
  const int tile_rank = (blockIdx.x / heads) * 4 + wave;
  if (tile_rank >= args.num_tiles) return;
  const int tile = tile_rank;                                // the list is sorted: longest first
  const int kvh = head_slot / args.head_blocks;
  const int hb = head_slot % args.head_blocks;
  const int entry = uniform(args.tiles[tile * 3]), tok0 = uniform(args.tiles[tile * 3 + 1]),
            ntok = uniform(args.tiles[tile * 3 + 2]);
  const int* table = a.table + (int64_t)entry * a.table_width;
  const int tq = 16 / args.rows_per_token;                   // tokens per 16-row tile

  const int ti = r / args.rows_per_token;
  const int hh = hb * 16 + r % args.rows_per_token;
  const int head = kvh * group + min(hh, group - 1);
  const int pos_first = uniform(a.positions[tok0]);          // positions are consecutive
  const int pos_last = pos_first + ntok - 1;
  const int lo_all = first_visible(a, pos_first);
  const float scale_log2 = a.scale * 1.44269504088896341f;

  TileState<HD> ts[TPW];
  int tile_first[TPW], tile_last[TPW], tile_lo[TPW], tile_lo_last[TPW];   // wave-uniform
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int t = j * tq + ti;
    // (16 rows need not be a whole number of tokens: a row past the tile's tokens would
    // be the next tile's token with this tile's key range, stored over the right result)
    const bool row_ok = ti < tq && t < ntok && hh < group;
    ts[j].pos = row_ok ? pos_first + t : -1;
    ts[j].lo = first_visible(a, ts[j].pos);
    ts[j].keep = a.keep;
    tile_first[j] = pos_first + j * tq;
    tile_last[j] = j * tq < ntok ? pos_first + min(ntok, (j + 1) * tq) - 1 : -1;
    tile_lo[j] = first_visible(a, tile_first[j]);
    tile_lo_last[j] = first_visible(a, tile_last[j]);
    load_query<HD>(ts[j], (const bf16_t*)a.q +
                   ((int64_t)(tok0 + min(t, ntok - 1)) * a.nq + head) * HD, row_ok, g);
  }

  const KeyWalk walk = key_walk<32>(a, lo_all);
  const int key_begin = walk.origin;
  PageCursor cur{(ConstTable)table, a.page_size, pos_last, walk, -1, -1};
  if (PAGE16) cur.start(key_begin);

  auto work = [&](const KvBlock<HD>& b, int v) {
    const int kb = walk.real(v);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if (kb > tile_last[j] || (kb + 31 < tile_lo[j] && kb >= a.keep)) continue;   // scalar conditions
      const bool interior = kb + 31 <= tile_first[j] && kb >= tile_lo_last[j];
      tile_update<HD>(ts[j], b, kb, scale_log2, interior, g);
    }
  };

  KvBlock<HD> A, B;
  load_kv_block<HD, PAGE16>(A, a, table, cur, kvh, key_begin, 32, r, g);
  for (int kb = key_begin; kb <= pos_last; kb += 64) {
    if (kb + 32 <= pos_last)
      load_kv_block<HD, PAGE16>(B, a, table, cur, kvh, kb + 32, 32, r, g);
    work(A, kb);
    if (kb + 32 > pos_last) break;
    if (kb + 64 <= pos_last)
      load_kv_block<HD, PAGE16>(A, a, table, cur, kvh, kb + 64, 32, r, g);
    work(B, kb + 32);
  }

#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const float sum = sum_with_sink(row_sum<HD>(ts[j]), ts[j].m, a.sink, head);        // by all lanes: it crosses lanes
    if (ts[j].pos < 0) continue;
    store_tile<HD>(ts[j], sum,
                   (bf16_t*)a.out + ((int64_t)(tok0 + j * tq + ti) * a.nq + head) * HD, g);
  }
}

#include "attention_prefill_lds_kernel.h"



// ---------------------------------------------------------------------------------
// The walk of the kernel above with the blocks brought into LDS by the memory system
// itself (head sizes 64 and 128, page sizes that are powers of two from 16 up).
//
// global_load_lds writes a wave's 64 x 16 bytes to consecutive LDS addresses, whatever
// global addresses the lanes name: each lane names the 16 bytes that its own operand
// register will hold, so the block lies in LDS in operand layout without passing through
// registers, nothing is selected or stored by the waves, and the loads of a block are
// issued two blocks ahead into a ring of three buffers at no cost in registers.  (Measured
// on the kernel above: bringing a block in through registers, one block ahead, is a
// third to two fifths of its time.)
//
// For the values to be 16 bytes per lane the keys of a block are assigned to the rows of
// the two score products so that a lane's eight scores belong to eight consecutive keys:
// row i of product b is key (i / 4) * 8 + b * 4 + i % 4 of the block.  Lane (r, g) then
// holds the scores of keys g * 8 .. g * 8 + 7 and needs V^T[d][those keys], one 16-byte
// run of a page's row.
//
// A page that is not there (beyond the context, or given back by a window) is read from
// page 0 instead: its scores are masked, their weights are exactly zero, and what the
// cache holds is finite.
// 64 x 16 bytes from the lanes' global addresses to LDS at `dst` + 16 * lane, without
// registers in between.  Written as an instruction rather than through the compiler's
// builtin: the compiler, knowing such a load writes LDS, makes LDS reads wait for every
// one of them in flight (it cannot always tell the buffers apart), which is the opposite
// of sending for blocks ahead of time.  The kernel counts these loads itself (s_waitcnt
// vmcnt) and separates them from the reads by a barrier; "memory" tells the compiler that
// LDS has changed.
__device__ __forceinline__ void lds_dma16(const void* src, void* dst) {
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)dst;
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(lds)
               : "memory", "m0");
}

// Steps of single tokens take it, and those in which single tokens are most of the work (a workgroup's four
// waves walk one request's keys with one row each in use, three workgroups a unit): there it waits for
// memory, and tiles of 32 rows, two workgroups a unit, are behind (136 entries of 300 tokens 29 against
// 34 us, 200 of 4,000 575 against 588).
template <int HD>
__global__ __launch_bounds__(256, 3) void attention_prefill_async_kernel(AttentionMfmaArgs args) {
  constexpr int KS = HD / 32, DB = HD / 16;
  constexpr int KQ = 2 * KS / 4, VQ = DB / 4;               // slots a wave brings in per block
  static_assert(HD % 64 == 0, "head sizes in steps of 64");
  // a ring buffer: the key slots of a block, then its value slots; three of them
  constexpr int kSlots = 2 * KS + DB;
  extern __shared__ __attribute__((aligned(16))) unsigned char prefill_lds[];
  typedef bf16x8 (*Slots)[kWave];
  const AttentionArgs& a = args.base;
  const int wave = uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;   // which of the item's four tiles
  const Slots ring = (Slots)prefill_lds;
  const int r = lane % 16, g = lane / 16;
  const int group = a.nq / a.nkv;
  const int heads = a.nkv * args.head_blocks;
  const int head_slot = blockIdx.x % heads;                   // one head per XCD's L2
  const int rank = blockIdx.x / heads;
  const int kvh = head_slot / args.head_blocks;
  const int hb = head_slot % args.head_blocks;
  const int P = a.page_size;
  const int tq = 16 / args.rows_per_token;
  const float scale_log2 = a.scale * 1.44269504088896341f;

  // Where this lane's 16 bytes of each slot lie, relative to the start of the half of the
  // block (16 keys) they belong to.  Keys: slot q = b * KS + s0 is product b, elements
  // g*8*KS + s0*8 .. + 7 of the key in row r.  Values: slot db is head elements
  // db*16 .. + 15, this lane's row r of them, keys g*8 .. + 7 of the block.
  const int64_t page_stride = (int64_t)a.nkv * P * HD;         // elements, keys and values alike
  const bf16_t* k_head = (const bf16_t*)a.k_pages + (int64_t)kvh * P * HD;
  const bf16_t* v_head = (const bf16_t*)a.v_pages + (int64_t)kvh * HD * P;
  const bool k_second = r >= 8;          // this lane's keys lie in the block's second 16
  const bool v_second = g >= 2;
  unsigned k_off[KQ], v_off[VQ];         // bytes
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int q = wave + 4 * i, b = q / KS, s0 = q % KS;
    const int key16 = ((r / 4) * 8 + b * 4 + r % 4) % 16;    // inside its half
    k_off[i] = 2u * (key16 * HD + g * 8 * KS + s0 * 8);
  }
#pragma unroll
  for (int i = 0; i < VQ; ++i)
    v_off[i] = 2u * (((wave + 4 * i) * 16 + r) * P + (g % 2) * 8);
  constexpr int kLoads = KQ + VQ;        // vector memory loads a wave has in flight per block

  const int entry = uniform(args.tiles[rank * 3]), tok0 = uniform(args.tiles[rank * 3 + 1]),
            ntok = uniform(args.tiles[rank * 3 + 2]);
  const int* table = a.table + (int64_t)entry * a.table_width;

  const int ti = wave * tq + r / args.rows_per_token;
  const int hh = hb * 16 + r % args.rows_per_token;
  const int head = kvh * group + min(hh, group - 1);
  const bool row_ok = r / args.rows_per_token < tq && ti < ntok && hh < group;
  const int pos_first = uniform(a.positions[tok0]);
  const int pos_last = pos_first + ntok - 1;
  const int lo_all = first_visible(a, pos_first);

  TileState<HD> t;
  t.pos = row_ok ? pos_first + ti : -1;
  t.lo = first_visible(a, t.pos);
  t.keep = a.keep;
  const int tile_first = pos_first + wave * tq;
  const int tile_last = wave * tq < ntok ? pos_first + min(ntok, (wave + 1) * tq) - 1 : -1;
  const int tile_lo = first_visible(a, tile_first);
  const int tile_lo_last = first_visible(a, tile_last);
  load_query<HD>(t, (const bf16_t*)a.q + ((int64_t)(tok0 + min(ti, ntok - 1)) * a.nq + head) * HD,
                 row_ok, g);

  // The item's blocks of 32 keys, numbered from its first.
  const KeyWalk walk = key_walk<32>(a, lo_all);
  const int key_begin = walk.origin;
  const int nblocks = ((pos_last - key_begin) >> 5) + 1;
  PageCursor cur{(ConstTable)table, P, pos_last, walk, -1, -1};
  cur.start(key_begin);
  // issue the loads of block j into ring buffer `to`; calls come in order of
  // j, as the cursor needs
  auto issue = [&](int j, int to) {
    const int v = key_begin + 32 * j, kb = walk.real(v);
    const int in0 = kb & (P - 1), in1 = (kb + 16) & (P - 1);
    const int64_t p0 = (int64_t)max(cur.next0, 0) * page_stride, p1 = (int64_t)max(cur.next1, 0) * page_stride;
    const bf16_t* kb0 = k_head + p0 + in0 * HD;
    const bf16_t* kb1 = k_head + p1 + in1 * HD;
    const bf16_t* vb0 = v_head + p0 + in0;
    const bf16_t* vb1 = v_head + p1 + in1;
    const char* kbase = (const char*)(k_second ? kb1 : kb0);
    const char* vbase = (const char*)(v_second ? vb1 : vb0);
    const Slots kdst = ring + to * kSlots, vdst = kdst + 2 * KS;
#pragma unroll
    for (int i = 0; i < KQ; ++i) lds_dma16(kbase + k_off[i], &kdst[wave + 4 * i][0]);
#pragma unroll
    for (int i = 0; i < VQ; ++i) lds_dma16(vbase + v_off[i], &vdst[wave + 4 * i][0]);
    cur.start(v + 32);
  };

  // One turn: block j is worked on out of ring buffer `from` while block j + 2 is sent
  // for into buffer `to`, which block j - 1 was read from.
  auto turn = [&](int j, int from, int to) {
    const int kb = walk.real(key_begin + 32 * j);
    // this wave's share of block j has arrived: at most block j + 1's loads are in flight
    if (j + 1 < nblocks) __builtin_amdgcn_s_waitcnt(0x0F70 | kLoads);
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    // Every wave's share of block j is in LDS, and every wave is through with block
    // j - 1.  The bare barrier: __syncthreads would first wait for every load in flight,
    // the younger block's among them.  The empty statements keep the compiler from
    // moving LDS reads across it.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // Only now may block j - 1's buffer be written: a wave that has nothing to do with a
    // block (outside its tile's window, or past its tile's last row) runs ahead of the
    // others by a whole turn, and loads sent for before the barrier could land while a
    // slower wave still reads that buffer.
    if (j + 2 < nblocks) issue(j + 2, to);
    if (j < nblocks && kb <= tile_last && (kb + 31 >= tile_lo || kb < a.keep)) {
      const Slots kcur = ring + from * kSlots, vcur = kcur + 2 * KS;
      KvBlock<HD> b;
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int s0 = 0; s0 < KS; ++s0) b.k[blk][s0] = kcur[blk * KS + s0][lane];
#pragma unroll
      for (int db = 0; db < DB; ++db) b.v[db] = vcur[db][lane];
      tile_update<HD, true, true>(t, b, kb, scale_log2, kb + 31 <= tile_first && kb >= tile_lo_last, g);
    }
  };

  // The query rows are waited for here, once (the empty statement uses them), and not at
  // their first use inside the loop, where the wait would be for every block in flight
  // as well; with them gone the vector memory counter counts the blocks' loads alone.
#pragma unroll
  for (int s0 = 0; s0 < KS; ++s0) asm volatile("" : "+v"(t.q[s0]));
  __builtin_amdgcn_s_waitcnt(0x0F70);
  if (nblocks > 0) issue(0, 0);
  if (nblocks > 1) issue(1, 1);
  // written out three times so that every turn's ring buffers are constants
  for (int j = 0; j < nblocks; j += 3) {
    turn(j, 0, 2);
    if (j + 1 < nblocks) turn(j + 1, 1, 0);
    if (j + 2 < nblocks) turn(j + 2, 2, 1);
  }

  const float sum = sum_with_sink(row_sum<HD>(t), t.m, a.sink, head);              // by all lanes: it crosses lanes
  if (row_ok)
    store_tile<HD>(t, sum, (bf16_t*)a.out + ((int64_t)(tok0 + ti) * a.nq + head) * HD, g);
}

// Query tiles per wavefront: as many as the register file holds accumulators for.
constexpr int tiles_per_wave(int hd) { return hd <= 32 ? 4 : (hd <= 64 ? 2 : 1); }

// Which kernel takes the long portions of head sizes 64 and 128 (so that tests reach each at small
// sizes).  2, as any other value: the rule below; 0: turns of 32 keys everywhere; 3, 4, 5: the kernel of 32
// rows a wavefront with one set, two and four.
static int g_prefill_variant = 2;
extern "C" void ts_attention_prefill_variant(int v) { g_prefill_variant = v; }

// What a step's portions are cut into: 16-row tiles per work item (the returned number) and, where
// the kernel of 32 rows a wavefront takes them, sets of wavefronts that split an item's keys (`sets`,
// else 0).  `q_lens` and `starts` are the entries' tokens and first positions, `reach` the keys that a
// query sees at most (0: all), `heads` the key/value heads (x blocks of 16 query heads); `extras`, the second
// entry point's: scores are more than scale times the product.
//
// The forms of that kernel: eight tiles an item in one set (two workgroups a unit, the best rate), eight
// tiles in two sets (half the time for a long item), four tiles in four sets (a quarter, for
// portions that would leave units without an item, at two thirds of the rate, since half as many rows share
// what the unit loads).  Beside them the kernel of 16 rows a wavefront (three workgroups a unit), for steps in
// which single tokens are most of the work: those wait for memory, and it is the fewer rows of an item and the
// more workgroups that count.  A step takes the form with the smallest estimate.
//
// An estimate is launch and first trips to memory, then its items handed out to the units of a head's
// share of the chip, longest first, each to the one that is free first, as the hardware does it; where a unit
// holds several workgroups, or has four items and more, the items' mean share of a unit or the longest
// item, whichever is more.  An item takes its turns of 64 keys (of a portion: the products', longer where units
// have items on end than alone; of a single token: the memory's, the same in every form) and a part of its own.
// The numbers are fitted to the times of 755 steps (prompts, and single tokens beside portions; 2 to 16 key/value
// heads of 64 and 128): the choice is the fastest form or within 4 per cent of it in 735, 0.4 per cent behind
// it in the mean; of 100 steps of random sizes that were timed afterwards in 98, 0.3.
// In us, one set / two / four / 16 rows: 16 and 8 heads of 128, 300 tokens 12.3 / 12.6 / 11.3 / 11.9, 2,048
// 47 / 40 / 36 / 50, 4,096 97 / 84 / 107 / 103, 8,192 286 / 303 / 382 / 370; 64 query heads, 8,192
// 1,009 / 1,136 / 1,410 / 1,326; 200 single tokens of 300 beside 33 tokens, 16 and 8 heads of 128
// 56 / 78 / 72 / 49, of 64 34 / 54 / 48 / 27; 400 of 1,500 beside 2,000
// 433 / 461 / 450 / 423 and 226 / 276 / 263 / 218.
namespace {
struct Item {
  int turns;        // of 64 keys
  bool single;      // of an entry of one token
};

// A step's items of so many tokens at most, longest first.
std::vector<Item> items_of(int tokens, int reach, int entries, const int* q_lens, const int* starts) {
  std::vector<Item> items;
  for (int e = 0; e < entries; ++e)
    for (int t = 0; t < q_lens[e]; t += tokens) {
      const int n = t + tokens < q_lens[e] ? tokens : q_lens[e] - t;
      int keys = starts[e] + t + n;
      if (reach > 0 && keys - n > reach) keys = reach + n;
      items.push_back({(keys + 63) / 64, q_lens[e] == 1});
    }
  std::stable_sort(items.begin(), items.end(), [](const Item& a, const Item& b) { return a.turns > b.turns; });
  return items;
}

// us of a form: `launch`; of a portion's item `item` and, a turn, `alone` or `together`; of a single token's
// `single` and `single_alone`.  Times of turns are at head size 128.
struct Form {
  double launch, item, alone, together, single, single_alone;
};
constexpr double kSingleTogether = 1.19;     // a single token's turn where its unit has others
constexpr Form kOneSet{5.2, 1.3, 1.42, 0.97, 2.0, 1.75}, kTwoSets{2.3, 4.45, 1.0, 1.12, 6.0, 0.94},
    kFourSets{0.0, 5.0, 0.81, 0.715, 4.5, 0.845}, kRows16{3.8, 0.86, 1.53, 0.64, 0.0, 1.55};

// The estimate's two kinds of times, by head size and by what makes a score.
struct Rates {
  double products, memory;
  double alone(const Form& f, const Item& i) const {
    return i.turns * (i.single ? f.single_alone * memory : f.alone * products);
  }
  double own(const Form& f, const Item& i) const { return i.single ? f.single : f.item; }
  double together(const Form& f, const Item& i) const {
    return own(f, i) + i.turns * (i.single ? kSingleTogether * memory : f.together * products);
  }
};

double mean_share(const Form& f, const Rates& r, const std::vector<Item>& items, int bins) {
  double sum = 0.0;
  for (const Item& i : items) sum += r.together(f, i);
  return sum / bins;
}

// Several workgroups a unit: `rest` of what is not the bound is not hidden behind it.
double side_by_side(const Form& f, const Rates& r, const std::vector<Item>& items, int bins, double rest) {
  double longest = 0.0;
  for (const Item& i : items) longest = std::max(longest, r.alone(f, i));
  const double share = mean_share(f, r, items, bins);
  return f.launch + std::max(longest, share) + rest * std::min(longest, share);
}

double handed_out(const Form& f, const Rates& r, const std::vector<Item>& items, int bins) {
  if ((int64_t)items.size() > 4 * (int64_t)bins) return f.launch + mean_share(f, r, items, bins);
  struct Unit {
    double us, shown;       // with every item's time together; with that of its only item alone
    bool operator<(const Unit& o) const { return us > o.us; }       // the heap's first is free first
  };
  std::vector<Unit> units(bins, Unit{0.0, 0.0});
  for (const Item& i : items) {
    std::pop_heap(units.begin(), units.end());
    Unit& u = units.back();
    const bool first = u.us == 0.0;
    u.us += r.together(f, i);
    u.shown = first ? r.own(f, i) + r.alone(f, i) : u.us;
    std::push_heap(units.begin(), units.end());
  }
  double most = 0.0;
  for (const Unit& u : units) most = std::max(most, u.shown);
  return f.launch + most;
}

int plan(int head_dim, int page_size, int rows_per_token, int heads, int reach, int entries, const int* q_lens,
         const int* starts, bool extras, int* sets) {
  *sets = 0;
  if (!(page_size >= 16 && (page_size & (page_size - 1)) == 0)) return tiles_per_wave(head_dim);
  if ((head_dim != 64 && head_dim != 128) || g_prefill_variant == 0) return 4;
  if (g_prefill_variant >= 3 && g_prefill_variant <= 5) {
    *sets = g_prefill_variant == 3 ? 1 : g_prefill_variant == 4 ? 2 : 4;
    return *sets == 4 ? 4 : 8;
  }
  if (entries <= 0 || *std::max_element(q_lens, q_lens + entries) <= 1) return 4;
  try {
    const int tokens16 = 16 / rows_per_token, bins = std::max(1, compute_units() / heads);
    const std::vector<Item> four = items_of(4 * tokens16, reach, entries, q_lens, starts),
                            eight = items_of(8 * tokens16, reach, entries, q_lens, starts);
    Rates tall = head_dim == 64 ? Rates{0.68, 0.57} : Rates{1.0, 1.0}, rows16 = tall;
    // (with scores of more than a product that kernel is another, at 128 half as fast: 200 single tokens of 300
    // beside 33 80 us, in one set 60; at 64 33 and 39)
    if (extras) tall.products *= 1.34, rows16.products *= 1.27, rows16.memory *= 1.24;
    const double us[] = {side_by_side(kOneSet, tall, eight, bins, 0.0), handed_out(kTwoSets, tall, eight, bins),
                         handed_out(kFourSets, tall, four, bins),
                         extras && head_dim == 128 ? HUGE_VAL : side_by_side(kRows16, rows16, four, bins, 0.28)};
    constexpr int kSets[] = {1, 2, 4, 0}, kTiles[] = {8, 8, 4, 4};
    const int best = (int)(std::min_element(us, us + 4) - us);
    *sets = kSets[best];
    return kTiles[best];
  } catch (const std::exception&) {      // no memory for the estimate: any step may take this kernel
    return 4;
  }
}
}  // namespace

extern "C" int ts_attention_prefill_plan(int head_dim, int page_size, int rows_per_token, int heads, int reach,
                                         int entries, const int* q_lens, const int* starts, int* sets) {
  return plan(head_dim, page_size, rows_per_token, heads, reach, entries, q_lens, starts, false, sets);
}
extern "C" int ts_attention_prefill_plan_scores(int head_dim, int page_size, int rows_per_token, int heads, int reach,
                                                int entries, const int* q_lens, const int* starts, int* sets) {
  return plan(head_dim, page_size, rows_per_token, heads, reach, entries, q_lens, starts, true, sets);
}

int launch_attention_prefill_tall(const AttentionMfmaArgs& args, hipStream_t stream);

template <int HD>
static int launch_prefill_lds(const AttentionMfmaArgs& args, hipStream_t stream) {
  if (args.tiles_per_wave != 4) TS_FAIL("attention_prefill: the LDS kernel takes items of 4 tiles");
  const int items = args.num_tiles * args.base.nkv * args.head_blocks;
  if constexpr (HD == 64 || HD == 128) {
    constexpr int lds = 3 * (2 * (HD / 32) + HD / 16) * kWave * 16;
    auto kernel = attention_prefill_async_kernel<HD>;
    static bool raised = false;     // per instantiation
    if (!raised) {
      if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        TS_FAIL("attention_prefill: cannot raise the LDS limit to %d bytes", lds);
      raised = true;
    }
    hipLaunchKernelGGL(kernel, dim3(items), dim3(256), lds, stream, args);
  } else {
    hipLaunchKernelGGL((attention_prefill_lds_kernel<HD>), dim3(items), dim3(256), 0, stream, args);
  }
  return 0;
}

template <int HD, bool PAGE16>
static int launch_prefill(const AttentionMfmaArgs& args, hipStream_t stream) {
  if (args.tiles_per_wave != tiles_per_wave(HD))
    TS_FAIL("attention_prefill: tiles_per_wave=%d, head size %d takes %d", args.tiles_per_wave,
            HD, tiles_per_wave(HD));
  dim3 grid(((args.num_tiles + 3) / 4) * args.base.nkv * args.head_blocks);
  hipLaunchKernelGGL((attention_prefill_kernel<HD, tiles_per_wave(HD), PAGE16>), grid, dim3(256),
                     0, stream, args);
  return 0;
}

int ts_check_attention_mfma_args(const AttentionMfmaArgs& args, const char* who);
int launch_attention_prefill_scores(const AttentionMfmaArgs& args, hipStream_t stream);

// `tiles` lists wave items (entry, first flat token, tokens) of at most
// tiles_per_wave * (16 / rows_per_token) consecutive tokens each.
extern "C" int ts_attention_prefill(const AttentionMfmaArgs* p, hipStream_t stream) {
  AttentionMfmaArgs args = *p;
  const AttentionArgs& a = args.base;
  if (a.num_tokens <= 0 || args.num_tiles <= 0) return 0;
  if (ts_check_attention_mfma_args(args, "attention_prefill")) return -1;
  if (!args.tiles) TS_FAIL("attention_prefill: no tile list");
  const bool page16 = a.page_size >= 16 && (a.page_size & (a.page_size - 1)) == 0;
  if (has_score_extras(a) && !page16)
    TS_FAIL("attention_prefill: scores with extras take pages of a power of two from 16");
  if (args.sets > 0) {
    if (!page16 || (a.hd != 64 && a.hd != 128) || args.tiles_per_wave != (args.sets == 4 ? 4 : 8))
      TS_FAIL("attention_prefill: %d sets of wavefronts with items of %d tiles, head size %d, pages of %d", args.sets,
              args.tiles_per_wave, a.hd, a.page_size);
    if (launch_attention_prefill_tall(args, stream)) return -1;
    TS_CHECK_LAUNCH("attention_prefill");
    return 0;
  }
  if (has_score_extras(a)) {
    if (args.tiles_per_wave != 4) TS_FAIL("attention_prefill: the LDS kernel takes items of 4 tiles");
    if (launch_attention_prefill_scores(args, stream)) return -1;
    TS_CHECK_LAUNCH("attention_prefill");
    return 0;
  }
  int rc = 0;
  switch (a.hd) {
#define TS_CASE(HD)                                                               \
  case HD:                                                                        \
    rc = page16 ? launch_prefill_lds<HD>(args, stream) : launch_prefill<HD, false>(args, stream); \
    break;
    TS_CASE(16) TS_CASE(32) TS_CASE(48) TS_CASE(64) TS_CASE(80) TS_CASE(96) TS_CASE(112)
    TS_CASE(128) TS_CASE(144) TS_CASE(160) TS_CASE(176) TS_CASE(192) TS_CASE(208) TS_CASE(224)
    TS_CASE(240) TS_CASE(256)
#undef TS_CASE
    default: TS_FAIL("attention_prefill: head_dim=%d not built", a.hd);
  }
  if (rc) return rc;
  TS_CHECK_LAUNCH("attention_prefill");
  return 0;
}
