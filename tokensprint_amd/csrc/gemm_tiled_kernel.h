// Matrix products of many rows (portions of prompts): C[M, N] = A[M, K] W[N, K]^T in
// bfloat16 with float32 sums, tiled through LDS for the matrix cores of gfx950.
//
// A workgroup of eight waves (two to a SIMD: one wave alone cannot keep a matrix core
// busy, its instructions issue at two thirds of the core's rate) owns a BM x BN tile of C
// and walks K in steps of 64.  Both
// operands are contiguous along K, which is also how a matrix-core instruction wants
// them (a lane holds eight consecutive k of one row), so a step's slab of A (BM rows of
// 128 bytes) and of W (BN rows) goes from global memory straight into LDS by
// `global_load_lds_dwordx4`, 16 bytes a lane, without passing through registers, several
// steps ahead in a ring of buffers; the waves count their own loads (s_waitcnt vmcnt),
// and one workgroup barrier a step separates the loads' arrival from the reads and the
// reads from the next overwrite.  A row's eight 16-byte pieces are stored in LDS at
// position (piece ^ (row / 2 % 8)), which makes the sixteen rows that a quarter wave reads
// together fall into different banks; since a direct load writes lane l's piece to slot
// l, the permutation is applied on the global side (which piece a lane fetches).
//
// The product is computed as C^T = W A^T (W's rows are the instruction's first operand),
// so a lane ends up with four consecutive columns of one row of C and stores them as one
// piece.  With PAIR, W is [2, N, K] (gate rows, then up rows): a tile holds BN/2 columns
// of each, interleaved per wave, and the epilogue writes silu(gate) * up.
//
// K is summed in index order by one accumulator per element whatever the tile size, so
// the choice of tile changes no bit of the result.
//
// Two further forms put the residual add and the RMSNorm of a prompt's step into the
// products around them, as the weight-streaming kernels do for few rows.  TAIL (the
// product that ends a sub-layer): stream += bfloat16(A W^T) in float32 in place, and the
// stream is handed on as `prepared` = bfloat16(stream * norm weight), not yet divided by
// the row's root mean square, with the rows' sums of squares in slices of 32 columns
// (`sumsq_out` [N / 32, M]; a slice is added up in the same order whatever the tile).
// SCALED (the product behind that norm): A is such prepared rows, and the epilogue
// multiplies row m by rsqrt(sum of its slices / K + eps), which a workgroup works out for
// its BM rows before it sends for its first operands.  HEADS is SCALED for a q/k/v projection with
// heads of as many elements as a tile has columns: the tile, rounded, passes LDS and leaves as
// qk_prepare.hip would have left it (normed and turned queries, keys and values in their pages).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_common.h"
#include "qk_prepare.h"

namespace {

struct TiledArgs {
  const bf16_t* a;
  const bf16_t* w;
  void* c;
  int M, N, K;          // N: columns of C (with PAIR: of each half of W)
  int tiles_m, tiles_n;
  int panel;            // tiles of a panel along M
  // SCALED: the sums of squares of A's rows [parts, M], or (`row_stride` not 0, a multiple of 4) a row's
  // side by side, as the weight-streaming tail form leaves them
  const float* sumsq_in;
  int parts, row_stride;
  float eps;
  // TAIL: the float32 stream [M, N] (read and written), the norm's weight [N], what is
  // handed on [M, N], the sums of squares of the new stream's rows [N / 32, M]
  float* resid;
  const float* norm_w;
  bf16_t* prepared;
  float* sumsq_out;
  float limit;          // PAIR: gated_unit's limit (0: silu, below: gelu)
};

// HEADS: `qkv`, `paged`, `store_kv` and `row_extra` of the preparation's arguments are not looked at.
struct TiledHeadsArgs : TiledArgs {
  QkPrepareArgs heads;
};

constexpr int kPlain = 0, kScaled = 1, kTail = 2, kHeads = 3;
constexpr int kSliceColumns = 32;   // columns per slice of a row's sum of squares (TAIL)

// One 16-byte piece per lane from global memory (uniform base + per-lane byte offset)
// into LDS at `lds` + 16 * lane.
__device__ __forceinline__ void dma16(const void* base, unsigned offset, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(offset), "s"(base), "s"(lds)
               : "memory", "m0");
}

template <int N>                                          // N: loads that may still be in flight
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "the load counter has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Rows of a tile's bfloat16 results in LDS, on their way out (HEADS): 16 bytes further from one another
// than they are long.
constexpr int kHeadRow = 128 + 8;

// HEADS: what becomes of one head of BM tokens from row m0 on.  `put` writes the tile into LDS, where
// sixteen lanes take a row, eight elements each, as qk_prepare.hip's do (the same sums in the same
// order), the tables' rows and pages asked for before the tile is there.  The preparation kernel read
// and wrote what the product had just written (50 MB and 9 us a layer of 2,048 rows of 4,096 columns);
// this is 1.7, 2.7 and 4.2 us at the end of a tile of 64, 128 and 256 rows (K = 1,024, against the same tile
// written as it is), of shuffles, LDS and the tables' trip.  Values go into their pages
// sixteen tokens at a time: where these fill a run of sixteen places (a prompt's mostly do), 16 bytes a
// lane, eight tokens of one element, else an element at a time.
template <int BM, int THREADS, typename PUT>
__device__ __forceinline__ void heads_out(const TiledHeadsArgs& g, int head, int m0, const int* row_pos,
                                          const int* row_entry, bf16_t* rows, PUT put) {
  constexpr int HD = 128, L = HD / 8, AT_ONCE = THREADS / L, TURNS = BM / AT_ONCE, AHEAD = TURNS < 4 ? TURNS : 4;
  static_assert(BM % AT_ONCE == 0 && TURNS % AHEAD == 0, "whole turns");
  const QkPrepareArgs& a = g.heads;
  const int sub = threadIdx.x % L, row0 = threadIdx.x / L;
  auto page_of = [&](int row) {
    return a.table[(int64_t)row_entry[row] * a.table_width + row_pos[row] / a.page_size];
  };
  if (head >= a.nq + a.nkv) {
    const int kvh = head - a.nq - a.nkv;
    __syncthreads();                                // the slabs have been read
    put(rows);
    __syncthreads();
    // 256 threads take sixteen tokens, sixteen lanes of them eight elements of each
    constexpr int TILES = THREADS / 256;            // of sixteen tokens at a time
    const int part = threadIdx.x / 16 % 16, lane = threadIdx.x % 16;
    for (int t0 = threadIdx.x / 256 * 16; t0 < BM; t0 += TILES * 16) {
      if (m0 + t0 >= g.M) break;
      const int row = t0 + lane, page = page_of(row), pos = row_pos[row];
      const int first = __shfl(pos, 0, 16), first_page = __shfl(page, 0, 16);
      const bool in_run = m0 + row < g.M && pos == first + lane && page == first_page &&
                          first % 16 == 0 && a.page_size % 16 == 0;
      const unsigned long long runs = __builtin_amdgcn_ballot_w64(in_run);
      bf16_t* pages = (bf16_t*)a.v_dst;
      if (runs == ~0ull) {
        if (first_page < 0) continue;
        bf16_t* dst = pages + ((int64_t)first_page * a.nkv + kvh) * a.page_size * HD + first % a.page_size;
        const int d = part * 8 + lane / 2, half = lane % 2 * 8;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = rows[(t0 + half + j) * kHeadRow + d];
        *(bf16x8*)(dst + (int64_t)d * a.page_size + half) = v;
      } else if (m0 + row < g.M && page >= 0) {
        bf16_t* dst = pages + ((int64_t)page * a.nkv + kvh) * a.page_size * HD + pos % a.page_size;
        const bf16x8 v = *(const bf16x8*)(rows + row * kHeadRow + part * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[(int64_t)(part * 8 + j) * a.page_size] = v[j];
      }
    }
    return;
  }
  const bool key = head >= a.nq;
  const float* w = key ? a.k_weight : a.q_weight;
  const bool first = sub < L / 2;
  float own_w[8], other_w[8];
  if (w) {
#pragma unroll
    for (int j = 0; j < 8; ++j) own_w[j] = w[sub * 8 + j], other_w[j] = w[(sub ^ (L / 2)) * 8 + j];
  }
  f32x4 cs[AHEAD][4];
  int page[AHEAD];
  auto fetch = [&](int u, int turn) {
    const int row = row0 + turn * AT_ONCE;
    if (a.cos) {
      const int64_t at = (int64_t)row_pos[row] * (HD / 2) + sub % (L / 2) * 8;
      cs[u][0] = *(const f32x4*)(a.cos + at);
      cs[u][1] = *(const f32x4*)(a.cos + at + 4);
      cs[u][2] = *(const f32x4*)(a.sin + at);
      cs[u][3] = *(const f32x4*)(a.sin + at + 4);
    }
    page[u] = key ? page_of(row) : 0;
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) fetch(u, u);
  __syncthreads();                                  // the slabs have been read
  put(rows);
  __syncthreads();
  for (int turn0 = 0; turn0 < TURNS; turn0 += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int row = row0 + (turn0 + u) * AT_ONCE;
      const bf16x8 x = *(const bf16x8*)(rows + row * kHeadRow + sub * 8);
      const bf16x8 y = *(const bf16x8*)(rows + row * kHeadRow + (sub ^ (L / 2)) * 8);
      float v[8], other[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (float)x[j], other[j] = (float)y[j];
      if (w) {
        const float rstd = head_rstd(v, L, HD, a.eps);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= rstd * own_w[j], other[j] *= rstd * other_w[j];
      }
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = (bf16_t)(a.cos ? head_turned(v[j], other[j], cs[u][j / 4][j % 4], cs[u][2 + j / 4][j % 4], first)
                              : v[j]);
      const int m = m0 + row;
      if (m < g.M) {
        if (!key) {
          *(bf16x8*)((bf16_t*)a.q_out + ((int64_t)m * a.nq + head) * HD + sub * 8) = o;
        } else if (page[u] >= 0) {
          *(bf16x8*)((bf16_t*)a.k_dst + (((int64_t)page[u] * a.nkv + head - a.nq) * a.page_size +
                                         row_pos[row] % a.page_size) * HD + sub * 8) = o;
        }
      }
      if (turn0 + AHEAD < TURNS) fetch(u, turn0 + AHEAD + u);
    }
  }
}

template <int FORM>
using TiledArgsOf = std::conditional_t<FORM == kHeads, TiledHeadsArgs, TiledArgs>;

template <int BM, int BN, int GM, int GN, int STAGES, bool PAIR, typename TO, int FORM = kPlain>
__global__ __launch_bounds__(64 * GM * GN, 1) void gemm_tiled_kernel(TiledArgsOf<FORM> g) {
  constexpr bool kRowScaled = FORM == kScaled || FORM == kHeads;
  static_assert(FORM != kHeads || (BN == 128 && !PAIR && BM * kHeadRow * 2 <= STAGES * (BM + BN) * 128),
                "a tile is one head of 128 elements, and has room in LDS");
  static_assert(!(FORM == kTail && PAIR), "the product that ends a sub-layer has one weight");
  constexpr int NW = GM * GN;                        // waves: GM along the rows, GN along the columns
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole load instructions per operand");
  constexpr int WM = BM / GM, WN = BN / GN;          // a wave's part of the tile
  static_assert(WM % 16 == 0 && WN % (PAIR ? 32 : 16) == 0, "a wave's part in 16 x 16 blocks");
  constexpr int TM = WM / 16, TN = WN / 16;
  static_assert(FORM != kTail || WN % kSliceColumns == 0, "a wave holds whole slices of a row");
  constexpr int LA = BM / (8 * NW), LW = BN / (8 * NW);   // load instructions a wave issues per step
  constexpr int LOADS = LA + LW;
  constexpr int STAGE_BYTES = (BM + BN) * 128;
  static_assert(STAGES >= 2 && STAGES <= 8, "a ring of 2 to 8 buffers");
  static_assert(LOADS * (STAGES - 1) < 64, "the load counter has six bits");
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiled_lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, gq = lane >> 4;
  const int wm = wave / GN, wn = wave % GN;

  // Which tile: workgroups go round the 8 XCDs by their index, each XCD has an L2 of its
  // own, so each XCD gets an eighth of the tiles that lie together (its workgroups share rows
  // of A and W): the tile grid is walked in panels of `panel` tiles along M, down a panel's
  // columns.
  const int local = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per_xcd + local;
  if (tile >= g.tiles_m * g.tiles_n) return;
  const int panel = tile / (g.panel * g.tiles_n), in_panel = tile - panel * g.panel * g.tiles_n;
  const int height = min(g.panel, g.tiles_m - panel * g.panel);
  const int tile_m = panel * g.panel + in_panel % height, tile_n = in_panel / height;
  const int m0 = tile_m * BM;

  // SCALED: the factors of this tile's rows.  Called once the first direct loads are on
  // their way and before the K loop counts loads: these loads are waited for with all
  // those before them, which the first turn needs anyway.  A row's slices are asked for
  // 32 at a time and added in their order.
  float* row_scale = (float*)(tiled_lds + STAGES * ((BM + BN) * 128));
  int* row_pos = (int*)(row_scale + BM);             // HEADS: position and entry of the tile's rows
  int* row_entry = row_pos + BM;
  auto row_scales = [&]() {
    if constexpr (kRowScaled) {
      for (int row = threadIdx.x; row < BM; row += 64 * NW) {
        const int m = min(m0 + row, g.M - 1);
        float sq = 0.f;
        for (int p0 = 0; p0 < g.parts; p0 += 32) {
          float part[32];
          if (g.row_stride == 0) {
#pragma unroll
            for (int i = 0; i < 32; ++i)
              part[i] = g.sumsq_in[(int64_t)min(p0 + i, g.parts - 1) * g.M + m];
          } else {
            const float* at = g.sumsq_in + (int64_t)m * g.row_stride;
#pragma unroll
            for (int i = 0; i < 32; i += 4) {
              const f32x4 four = *(const f32x4*)(at + min(p0 + i, g.row_stride - 4));
#pragma unroll
              for (int e = 0; e < 4; ++e) part[i + e] = four[e];
            }
          }
#pragma unroll
          for (int i = 0; i < 32; ++i) sq += p0 + i < g.parts ? part[i] : 0.f;
        }
        row_scale[row] = rsqrtf(sq / (float)g.K + g.eps);
        if constexpr (FORM == kHeads) {
          row_pos[row] = g.heads.positions[m];
          row_entry[row] = g.heads.entry_of_token[m];
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  };

  // TAIL with a small part of the tile per wave: the stream's values and the norm's
  // weights are asked for behind the last direct loads, a ring's length of K steps before
  // the epilogue that takes them out of registers (EARLY loads a lane, which the waits for
  // the last steps count).  Asked for before the first direct loads they were 8 MB of 2,048
  // rows of 1,024 that every tile waited for with its first step (23.1 us a product, 22.0 so).
  constexpr bool kEarlyStream = FORM == kTail && TM * TN <= 16;
  constexpr int EARLY = kEarlyStream ? TN * TM + TN : 0;
  static_assert(LOADS * (STAGES - 2) + EARLY < 64, "the load counter has six bits");
  f32x4 early_x[kEarlyStream ? TN : 1][kEarlyStream ? TM : 1], early_w[kEarlyStream ? TN : 1];
  auto early_loads = [&]() {
    if constexpr (kEarlyStream) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const int n = min(tile_n * BN + wn * WN + tn * 16 + gq * 4, g.N - 4);
        early_w[tn] = *(const f32x4*)(g.norm_w + n);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
          const int m = min(m0 + wm * WM + tm * 16 + r, g.M - 1);
          early_x[tn][tm] = *(const f32x4*)(g.resid + (int64_t)m * g.N + n);
        }
      }
    }
  };

  // row of the tile that LDS row `j` of the A slab holds: the upper halves of all waves' parts,
  // then the lower ones, where a turn takes them apart
  auto a_row = [&](int j) {
    if constexpr (TM * TN > 16) {
      const int in = j % (BM / 2);
      return in / (WM / 2) * WM + j / (BM / 2) * (WM / 2) + in % (WM / 2);
    } else {
      return j;
    }
  };
  // column of W (row of the stacked weight) that LDS row `j` of the W slab holds
  auto w_row = [&](int j) {
    if constexpr (PAIR) {
      const int half = j / WN, in = j % WN;           // which wave column, where in it
      const int col = tile_n * (BN / 2) + half * (WN / 2) + in % (WN / 2);
      return min(col, g.N - 1) + (in >= WN / 2 ? g.N : 0);
    } else {
      return min(tile_n * BN + j, g.N - 1);
    }
  };

  // per-lane byte offsets of this wave's loads: instruction i covers LDS rows
  // (NW i + wave) * 8 .. + 7 of the slab, lane l the piece at slot l % 8 of row l / 8
  unsigned off_a[LA], off_w[LW];
  const unsigned row_bytes = (unsigned)g.K * 2;
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int row = (NW * i + wave) * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ ((row >> 1) & 7);
    off_a[i] = (unsigned)min(m0 + a_row(row), g.M - 1) * row_bytes + piece * 16;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (NW * i + wave) * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ ((row >> 1) & 7);
    off_w[i] = (unsigned)w_row(row) * row_bytes + piece * 16;
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)tiled_lds;

  // load instruction i of this wave for K step kt into ring buffer `stage`
  auto issue_one = [&](int stage, int kt, int i) {
    const unsigned dst = lds0 + stage * STAGE_BYTES + wave * 1024;
    if (i < LA) dma16((const char*)g.a + (int64_t)kt * 128, off_a[i], dst + i * NW * 1024);
    else dma16((const char*)g.w + (int64_t)kt * 128, off_w[i - LA], dst + BM * 128 + (i - LA) * NW * 1024);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = f32x4{0.f, 0.f, 0.f, 0.f};

  // a lane's reads: row r of a 16-row block, the piece that holds k = 32 ks + 8 gq ..
  const int swz = (r >> 1) & 7;
  const int read0 = r * 128 + ((gq ^ swz) << 4), read1 = r * 128 + (((4 + gq) ^ swz) << 4);

  struct Frags {
    bf16x8 a[TM], w[TN];
  };
  auto read = [&](Frags& f, int stage, int ks) {
    const unsigned char* slab = tiled_lds + stage * STAGE_BYTES;
    const unsigned char* sa = slab + wm * WM * 128 + (ks ? read1 : read0);
    const unsigned char* sw = slab + (BM + wn * WN) * 128 + (ks ? read1 : read0);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) f.w[tn] = *(const bf16x8*)(sw + tn * 2048);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) f.a[tm] = *(const bf16x8*)(sa + tm * 2048);
  };
  // the products of one K step of 32; with `load` the wave's loads for K step `kt` are
  // issued between them, so that neither the matrix cores nor the loads' issue wait
  auto mma = [&](const Frags& f, auto with_loads, int stage, int kt) {
    constexpr bool load = decltype(with_loads)::value;
    constexpr int EVERY = (TN * TM) / LOADS > 0 ? (TN * TM) / LOADS : 1;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[tn], f.a[tm], acc[tn][tm], 0, 0, 0);
        const int idx = tn * TM + tm;
        if constexpr (load) {
          if (idx % EVERY == 0 && idx / EVERY < LOADS) issue_one(stage, kt, idx / EVERY);
        }
      }
    if constexpr (load) {
#pragma unroll
      for (int i = (TN * TM + EVERY - 1) / EVERY; i < LOADS; ++i) issue_one(stage, kt, i);
    }
  };

  // The ring: K step kt lives in buffer kt % STAGES.  A turn multiplies step kt's first
  // half while its second half comes out of LDS, then (after the barrier that says step
  // kt + 1 has arrived and step kt has been read by everyone) its second half while the
  // first half of step kt + 1 comes out of LDS and the loads of step kt + STAGES go out
  // into the buffer that step kt has left.
  const int KT = g.K / 64;                              // at least STAGES (the launcher's check)
  if constexpr (TM * TN > 16) {
    // A wave's part is too large to hold two K steps' operands beside its sums.  A turn (one K
    // step) is walked in blocks of TN products, a row block of A against the wave's columns:
    // the upper half of its row blocks with the first 32 of K, with the second, then the lower
    // half.  The columns' operands stay in registers for the turn, a row block's comes out of
    // LDS H blocks before its products, also across the turns' border.  So a step's W and
    // upper A have been read an eighth of a turn after their first use, its lower A an eighth
    // after its own, and two meetings a turn say so: the loads that go into their places have
    // about a turn to arrive with two buffers, and no wave waits for LDS in front of its products.
    // (With one meeting a turn, at its border, everything was waited for there and every half
    // began with a trip to LDS.  256 x 256 tiles, products of zeros, 2,048 x 24,576 x 4,096: 285 ->
    // 232 us, of ordinary data, where the card's power holds it back, 333 -> 314; 8,192 x 51,200 x
    // 5,120 3,986 -> 3,124, of that 125 by panels of eight tiles instead of four.  Four wavefronts
    // of 128 x 128, with two thirds of the reads of LDS, are as fast; a higher priority of half the
    // wavefronts, or of the products, changes nothing.)
    static_assert(STAGES == 2 && TM % 2 == 0 && LA % 2 == 0, "two buffers, whole halves of A");
    constexpr int H = TM / 2, LOWER = LA / 2, FIRST = LW + LOWER;
    // Load i of a step: the columns, the upper half of the rows, then the lower half.  A unit
    // takes a load in about 28 cycles, so a turn's are spread over its blocks, from block H on
    // (where the places of the first are free) and through block H - 1 of the next turn.
    auto issue = [&](int stage, int kt, int i) {
      issue_one(stage, kt, i < LW ? LA + i : i - LW);
    };
    auto at = [](int i) constexpr { return i * (4 * H) / LOADS; };   // blocks behind block H
    auto issued_before = [at](int q) constexpr {                     // of a step's loads
      int n = 0;
      for (int i = 0; i < LOADS; ++i) n += at(i) < q;
      return n;
    };
    static_assert(at(FIRST) >= 2 * H, "a place is free when it is sent for");
    constexpr int EARLY_LOADS = issued_before(3 * H), BY_MEETING = issued_before(2 * H);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) issue(0, 0, i);
#pragma unroll
    for (int i = 0; i < EARLY_LOADS; ++i) issue(1, 1, i);
    row_scales();
    auto meet = [&](auto in_flight) {
      __builtin_amdgcn_sched_barrier(0);
      wait_loads<decltype(in_flight)::value>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8 fw[2][TN], fa[H];
    auto read_columns = [&](int stage, int ks) {
      const unsigned char* sw = tiled_lds + stage * STAGE_BYTES + (BM + wn * WN) * 128 + (ks ? read1 : read0);
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) fw[ks][tn] = *(const bf16x8*)(sw + tn * 2048);
    };
    auto read_rows = [&](int stage, int half, int ks, int t) {
      fa[t] = *(const bf16x8*)(tiled_lds + stage * STAGE_BYTES +
                               (half * (BM / 2) + wm * (WM / 2) + t * 16) * 128 + (ks ? read1 : read0));
    };
    meet(std::integral_constant<int, LOWER + EARLY_LOADS>{});
    read_columns(0, 0);
#pragma unroll
    for (int t = 0; t < H; ++t) read_rows(0, 0, 0, t);
    // behind: steps that follow this one (2: two or more)
    auto turn = [&](auto steps_behind, int s, int kt) {
      constexpr int behind = decltype(steps_behind)::value;
      read_columns(s, 1);
#pragma unroll
      for (int b = 0; b < 4 * H; ++b) {
        const int half = b / (2 * H), ks = b / H % 2, t = b % H;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          acc[tn][half * H + t] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[ks][tn], fa[t], acc[tn][half * H + t], 0, 0, 0);
        // the lower half of this step has arrived; its W and upper half have been read
        if (b == H) meet(std::integral_constant<int, behind >= 1 ? LOADS : 0>{});
        if constexpr (behind >= 1) {
          // the next step's W and upper half have arrived; this one's lower half has been read
          if (b == 3 * H) {
            meet(std::integral_constant<int, behind >= 2 ? LOWER + BY_MEETING : LOWER>{});
            read_columns(s ^ 1, 0);
          }
        }
        if (b < 3 * H) read_rows(s, (b + H) / (2 * H), (b + H) / H % 2, t);
        else if constexpr (behind >= 1) read_rows(s ^ 1, 0, 0, t);
        if constexpr (behind >= 1) {
#pragma unroll
          for (int i = 0; i < LOADS; ++i) {
            if (b < H && at(i) == 3 * H + b) issue(s ^ 1, kt + 1, i);
            if (behind >= 2 && b >= H && at(i) == b - H) issue(s, kt + 2, i);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int kt = 0;
    for (; kt + 2 < KT; ++kt) turn(std::integral_constant<int, 2>{}, kt & 1, kt);
    turn(std::integral_constant<int, 1>{}, kt & 1, kt);
    turn(std::integral_constant<int, 0>{}, (kt + 1) & 1, kt + 1);
  } else {
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) issue_one(s, s, i);
  row_scales();
  wait_loads<LOADS * (STAGES - 1)>();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
  read(f0, 0, 0);
  // a turn's middle: step kt + 1 has arrived when at most IN_FLIGHT loads are on their way
  auto next_step = [&](auto in_flight, int stage) {
    wait_loads<decltype(in_flight)::value>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // this wave has read step kt
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(f0, stage, 0);
  };
  for (int kt0 = 0; kt0 < KT - STAGES; kt0 += STAGES) {
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
      const int kt = kt0 + s;
      if (kt < KT - STAGES) {
        read(f1, s, 1);
        mma(f0, std::false_type{}, 0, 0);
        next_step(std::integral_constant<int, LOADS * (STAGES - 2)>{}, (s + 1) % STAGES);
        mma(f1, std::true_type{}, s, kt + STAGES);
      }
    }
  }
  // the last STAGES turns, for which nothing is sent any more: written out, so that the turns
  // before them have one wait and no branch (2,048 x 2,048 x 2,048 in 128 x 128 tiles 22.1 ->
  // 19.6 us, 2,048 x 1,024 x 2,048 in 128 x 64 13.0 -> 12.6)
  early_loads();
  // (they have to lie in front of the waits that count them)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  const int last = (KT - STAGES) % STAGES;
  auto last_turn = [&](auto turn) {
    constexpr int t = decltype(turn)::value;
    const int stage = (last + t) % STAGES;
    read(f1, stage, 1);
    mma(f0, std::false_type{}, 0, 0);
    if constexpr (t + 1 < STAGES)
      next_step(std::integral_constant<int, LOADS * (STAGES - 2 - t) + EARLY>{}, (last + t + 1) % STAGES);
    mma(f1, std::false_type{}, 0, 0);
  };
  last_turn(std::integral_constant<int, 0>{});
  last_turn(std::integral_constant<int, 1>{});
  if constexpr (STAGES > 2) last_turn(std::integral_constant<int, 2>{});
  if constexpr (STAGES > 3) last_turn(std::integral_constant<int, 3>{});
  static_assert(STAGES <= 4, "the last turns are written out");
  }

  // acc[tn][tm][e] = C[m0 + wm WM + 16 tm + r][column block tn, column 4 gq + e]
  if constexpr (FORM == kTail) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int m = m0 + wm * WM + tm * 16 + r;
#pragma unroll
      for (int p = 0; p < TN / 2; ++p) {
        // a slice of 32 columns: this lane's four columns of the first block of sixteen in
        // order, those of the second, then the four lanes that share the row
        const int n_slice = tile_n * BN + wn * WN + p * kSliceColumns;
        const bool ok = m < g.M && n_slice < g.N;       // N is a multiple of 32 here
        float sq = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int n = n_slice + h * 16 + gq * 4;
          if (ok) {
            const int64_t at = (int64_t)m * g.N + n;
            f32x4 x, w4;
            if constexpr (kEarlyStream) {
              x = early_x[2 * p + h][tm];
              w4 = early_w[2 * p + h];
            } else {
              x = *(const f32x4*)(g.resid + at);
              w4 = *(const f32x4*)(g.norm_w + n);
            }
            bf16x4_t handed;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              // the product rounded to the activation type first, as the unfused path stores it
              x[e] += (float)(bf16_t)acc[2 * p + h][tm][e];
              sq += x[e] * x[e];
              handed[e] = (bf16_t)(x[e] * w4[e]);
            }
            *(f32x4*)(g.resid + at) = x;
            *(bf16x4_t*)(g.prepared + at) = handed;
          }
        }
        sq += __shfl_xor(sq, 16, 64);
        sq += __shfl_xor(sq, 32, 64);
        if (ok && gq == 0) g.sumsq_out[(int64_t)(n_slice / kSliceColumns) * g.M + m] = sq;
      }
    }
    return;
  }
  TO* c = (TO*)g.c;
  const bool clamped = PAIR && g.limit > 0.f;
  const float top = clamped ? g.limit : INFINITY, lift = clamped ? 1.f : 0.f;
  // the weight exp2(gc (slope + cubic gc^2)): of the sigmoid, or, for gelu_tanh(g) =
  // g sigmoid(2 sqrt(2 / pi) (g + 0.044715 g^3)), of that one
  const bool gelu = PAIR && g.limit < 0.f;
  const float slope = clamped ? -1.702f * 1.44269504f
                              : (gelu ? -1.59576912160573f * 1.44269504f : -1.44269504f);
  const float cubic = gelu ? 0.044715f * slope : 0.f;
  if constexpr (kRowScaled) {
    // (the barriers of the K loop lie between the factors' writes and these reads)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const float scale = row_scale[wm * WM + tm * 16 + r];
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[tn][tm][e] *= scale;
    }
  }
  if constexpr (FORM == kHeads) {
    heads_out<BM, 64 * NW>(g, tile_n, m0, row_pos, row_entry, (bf16_t*)tiled_lds, [&](bf16_t* rows) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          bf16x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (bf16_t)acc[tn][tm][e];
          *(bf16x4_t*)(rows + (wm * WM + tm * 16 + r) * kHeadRow + wn * WN + tn * 16 + gq * 4) = v;
        }
    });
    return;
  }
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
    const int m = m0 + wm * WM + tm * 16 + r;
    if (m >= g.M) continue;
    if constexpr (PAIR) {
#pragma unroll
      for (int tn = 0; tn < TN / 2; ++tn) {
        const int n = tile_n * (BN / 2) + wn * (WN / 2) + tn * 16 + gq * 4;
        if (n >= g.N) continue;
        const f32x4 gate = acc[tn][tm], up = acc[tn + TN / 2][tm];
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // as the separate kernel does it: the product rounded to the activation type first
          const float gv = (float)(TO)gate[e], uv = (float)(TO)up[e];
          // 64 values a lane at the very end of the kernel, the matrix cores idle: the
          // hardware's exp2 and reciprocal (an ulp each) instead of a division's ten steps
          // (gated_unit's three forms: the clamps change nothing without a limit; far on the
          // gate's negative side the power is infinite and the reciprocal zero)
          const float gc = fminf(gv, top), uc = fminf(fmaxf(uv, -top), top) + lift;
          const float power = gc * fmaf(cubic, gc * gc, slope);
          o[e] = gc * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(power)) * uc;
        }
        store4<TO>(c + (int64_t)m * g.N + n, o, g.N - n);
      }
    } else {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const int n = tile_n * BN + wn * WN + tn * 16 + gq * 4;
        if (n >= g.N) continue;
        store4<TO>(c + (int64_t)m * g.N + n, acc[tn][tm], g.N - n);
      }
    }
  }
}

template <int BM, int BN, int GM, int GN, int STAGES, bool PAIR, typename TO, int FORM>
int launch_tiled(TiledArgsOf<FORM> g, hipStream_t stream) {
  auto kernel = gemm_tiled_kernel<BM, BN, GM, GN, STAGES, PAIR, TO, FORM>;
  constexpr int lds = STAGES * (BM + BN) * 128 + (FORM == kScaled ? BM * 4 : FORM == kHeads ? BM * 12 : 0);
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static bool raised[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64)
    TS_FAIL("gemm_tiled: no current device below 64");
  if (!raised[device]) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) !=
        hipSuccess)
      TS_FAIL("gemm_tiled: %d bytes of LDS refused", lds);
    raised[device] = true;
  }
  if (g.K / 64 < STAGES) TS_FAIL("gemm_tiled: K=%d is too short for %d buffers", g.K, STAGES);
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + (PAIR ? BN / 2 : BN) - 1) / (PAIR ? BN / 2 : BN);
  // the height of a panel: the one with which the tiles that an XCD's units hold at a time (32)
  // bring the fewest rows of A and W into its L2.  (Regions of the grid, one an XCD, came before
  // it: where they divided the tiles unevenly one XCD had a round more than the others.
  // 1,536 x 10,304 x 2,048 in 246 tiles of 256 x 256: 92 -> 58 us.)
  const int per_xcd = (int)(((int64_t)g.tiles_m * g.tiles_n + 7) / 8), held = per_xcd < 32 ? per_xcd : 32;
  int64_t best_rows = -1;
  for (int p = 1; p <= 16; p *= 2) {
    const int64_t rows = (int64_t)(p < g.tiles_m ? p : g.tiles_m) * BM + (int64_t)((held + p - 1) / p) * BN;
    if (best_rows < 0 || rows < best_rows) { best_rows = rows; g.panel = p; }
  }
  hipLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(64 * GM * GN), lds, stream, g);
  TS_CHECK_LAUNCH("gemm_tiled");
  return 0;
}

// The tile that a product of these sizes takes when the caller names none: the one with
// the smallest estimate of rounds x time of a tile, a round being one tile on every
// compute unit.  A tile's time is a fixed part (launch, first loads, epilogue and the
// stores' way to memory; the SiLU of the paired form on top) and a part per K step of 64,
// both fitted to an MI355X at 65 to 8,192 rows of 23 weights (N 1,024 to 51,200, K 1,024 to
// 25,600) in memory, where the estimate's choice is the fastest tile but for 0.02 % of the time:
// a large tile needs fewer bytes from L2 per product and its steps are bound by the matrix cores
// (1.1 us for 256 x 256 on average; at what the card's power allows with all units busy on
// ordinary data up to 1.5, with zeros 1.2), a small one's by the rate at which a unit takes
// direct loads (0.33 us for 128 x 64, 2.3 times the matrix cores' time), but a tile is one
// workgroup and a unit without one idles.
// The tiles of 64 rows are for portions of few rows.  With 128 x 64 as the smallest, 300 rows of 1,024
// columns were 48 workgroups; the product that ends a sub-layer took 12.4 us with K = 2,048 and 16.6 with
// K = 3,072, and takes 7.3 and 9.5 in 64 x 32 tiles (160 workgroups of four wavefronts); 1,024 rows 13.2 and
// 18.0, in 64 x 64 tiles 10.3 and 13.5.  64 x 128 is for up to 64 rows of many columns, where a tile of 128
// rows brings every row of A twice (64 rows of 151,936 columns of 4,096: 244 us, 243 and 267 in 128 x 128
// and 128 x 64; 16 rows 224, 236, 242), and for rows that leave most of a last tile of 128 empty (192 rows of
// 10,240 columns: 240 tiles, 320 of 128 x 64).  Their fixed parts are what 65 to 1,024 rows of 21 weights show, and
// make a second round as long as the first, which for tiles that share a unit it is not (so the
// larger tiles are chosen there, which are about as fast).
struct TileCost {
  int tile, bm, bn;
  float fixed_us, step_us, pair_us;
};
constexpr TileCost kTileCosts[] = {
    {8, 64, 32, 2.2f, 0.1375f, 0.5f}, {7, 64, 64, 2.9f, 0.18f, 0.5f}, {3, 128, 64, 1.2f, 0.329f, 0.5f},
    {6, 64, 128, 1.2f, 0.329f, 0.5f}, {2, 128, 128, 2.4f, 0.491f, 0.8f}, {1, 256, 128, 4.5f, 0.721f, 1.4f},
    {5, 256, 192, 6.6f, 0.931f, 1.1f}, {4, 256, 256, 7.7f, 1.126f, 1.6f},
};

// (`least_rows`: of the tiles with so many rows or more)
inline int cheapest_tile(const TiledArgs& g, bool pair, int least_rows = 0) {
  const int units = compute_units();
  const int64_t cols = pair ? 2 * (int64_t)g.N : g.N;
  int best = 3;
  float best_us = -1.f;
  for (const TileCost& t : kTileCosts) {
    if (t.bm < least_rows) continue;
    const int64_t tiles = (int64_t)((g.M + t.bm - 1) / t.bm) * ((cols + t.bn - 1) / t.bn);
    const int64_t rounds = (tiles + units - 1) / units;
    const float us = rounds * (t.fixed_us + (pair ? t.pair_us : 0.f) + t.step_us * (g.K / 64));
    if (best_us < 0.f || us < best_us) { best_us = us; best = t.tile; }
  }
  return best;
}

template <bool PAIR, typename TO, int FORM = kPlain>
int choose_tile(const TiledArgs& g, int tile, hipStream_t stream) {
  if (tile == 0) tile = cheapest_tile(g, PAIR);
  switch (tile) {
    case 1: return launch_tiled<256, 128, 4, 2, 3, PAIR, TO, FORM>(g, stream);
    case 2: return launch_tiled<128, 128, 2, 4, 4, PAIR, TO, FORM>(g, stream);
    case 3: return launch_tiled<128, 64, 4, 2, 4, PAIR, TO, FORM>(g, stream);
    case 4: return launch_tiled<256, 256, 2, 4, 2, PAIR, TO, FORM>(g, stream);
    case 5: return launch_tiled<256, 192, 4, 2, 2, PAIR, TO, FORM>(g, stream);
    case 6: return launch_tiled<64, 128, 2, 4, 4, PAIR, TO, FORM>(g, stream);
    case 7: return launch_tiled<64, 64, 4, 2, 4, PAIR, TO, FORM>(g, stream);
    case 8: return launch_tiled<64, 32, 4, 1, 4, PAIR, TO, FORM>(g, stream);
  }
  TS_FAIL("gemm_tiled: no tile %d", tile);
}

}  // namespace
