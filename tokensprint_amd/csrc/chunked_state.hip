// Recurrences over a matrix S (N x P) per head,
//
//   S <- g S;   u = vs v   or   u = beta (vs v - S^T k);   S <- S + k u^T;   o = S^T q,
//
// for portions of many tokens: in chunks of 64 tokens whose inside is products of matrices, on
// the float32 matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, float32 sums).  With
// D(t) the product of the decays from the chunk's first token through t and M(t, s) the one
// from s + 1 through t, inside a chunk that starts from S0
//
//   o_t = D(t) S0^T q_t + sum_(s <= t) M(t, s) (q_t . k_s) u_s
//   S   = D(last) S0 + sum_s M(last, s) k_s u_s^T
//
// and the delta rule's u solve a unit triangular system,
//
//   u_t + beta_t sum_(s < t) M(t, s) (k_t . k_s) u_s = beta_t v_t - beta_t D(t) S0^T k_t,
//
// whose solution is Y - W S0 with Y and W that do not know S0.  So there are three launches (or, for
// linear forms in portions that are not too long, two: chunk_prepare and chunk_scan, below):
//   * every chunk by itself: its contribution to S (linear forms: chunk_local), or Y, W and the
//     decayed keys (delta rule: chunk_solve);
//   * the chunks of an entry in order: the state in front of each (chunk_carry, a multiply-add
//     an element; chunk_walk, two products a chunk for sixteen columns of S, which a workgroup
//     keeps in registers) and the state that the portion leaves;
//   * every chunk by itself: o (chunk_output).
//
// Decays are multiplied up, never divided and never taken through logarithms, so a decay of
// zero or one is as good as any other.  With a decay per row of S the products q . k and k . k
// carry a decay in every term: between blocks of 16 tokens it is split at the later block's
// first token into a factor on each side (both products of decays in between, at most one),
// inside a block it is multiplied up pair by pair.
//
// What bounds them: the float32 matrix rate (64 operations a cycle and SIMD) and, in chunk_walk,
// the chain of two products and two meetings in LDS a chunk.  The kernels before these walked a
// token at a time (the linear forms in chunks side by side, twice the arithmetic) and were bound
// by the chain of a token's multiply-adds and sums.  At 2,048 tokens, before and now (alone; in
// brackets the launches as they run in a prompt's step): delta rule, 16 heads of 128 x 128, 592 and
// 125 us (solve 31, walk 61, output 33); 8 heads of 64 x 128 with a decay per row 469 and 76 (21,
// 36, 19); fixed decays, 16 heads of 128 x 128, 230 and 78 (local 29, carry 22, output 44); state
// space, 64 heads of 128 x 64, 386 and 123 (41, 31, 67), in two launches 102 (25, 77).  The short
// chains of product_step and the decays in 64 bits are 1 to 10 us of that.
//
// Matrix operands: lane (g, l) = (lane / 16, lane % 16) holds row l of A, column l of B, and rows
// 4 g + r, column l of the sum.  The four steps of a 16-deep product take k = 4 g + r in step r
// (the same permutation of k on both sides), so four steps' operands are one 16-byte read, and
// a sum's registers are the B operands of a product over its rows.  Scratch is laid out in that
// order, so every access to it is 16 bytes a lane, side by side.
#include "chunked_state.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTok = kChunkTokens;         // tokens of a chunk
constexpr int kThreads = 256;
constexpr int kTileLd = 20;                // row of a 16 x 16 tile in LDS (16-byte reads, no conflicts)
constexpr int kTile = 16 * kTileLd;
// What happens to q, k (and v) on their way in: nothing, SiLU (v too), the rotation.
constexpr int kPlain = 0, kSilu = 1, kTurned = 2;
constexpr int kTiles = 10;                 // tiles on and below the diagonal of a 64 x 64 matrix

__device__ __forceinline__ float silu(float v) { return v / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus(float v) { return v > 20.f ? v : log1pf(expf(v)); }

// One of the four steps of a product of 16 by itself, to be added to others: the even and the odd
// steps are a chain of eight products each.  An element's error is mostly that of its chains and
// of the decays that it is multiplied with: 600 tokens, outputs of the delta rule (128 rows) off by
// 1.40e-7 of themselves, 1.58 in chains of sixteen with decays in 32 bits, 3.4 in one chain, 1.40
// walked; a decay per row and 64 rows 1.33, 1.54, 2.6, 1.35; fixed decays (128) 1.03, 1.24 (1.06 in
// chunks of multiply-adds); state space (128) 1.07, 1.22 (1.15).
__device__ __forceinline__ void product_step(f32x4 (&chain)[2], f32x4 a, f32x4 b, int r) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  chain[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], r < 2 ? zero : chain[r & 1], 0, 0, 0);
}
__device__ __forceinline__ f32x4 product2(f32x4 a, f32x4 b) {
  f32x4 chain[2];
#pragma unroll
  for (int r = 0; r < 4; ++r) product_step(chain, a, b, r);
  return chain[0] + chain[1];
}
// The same with every step a chain of its own, where few products are made or many results hang on
// one: the products of keys and queries, the triangular systems.
__device__ __forceinline__ f32x4 product4(f32x4 a, f32x4 b) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 step[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) step[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], zero, 0, 0, 0);
  return (step[0] + step[1]) + (step[2] + step[3]);
}
__device__ __forceinline__ f32x4 read4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void write4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ int tri(int i, int j) { return i * (i + 1) / 2 + j; }
__device__ __forceinline__ int tri_row(int t) { return t >= 6 ? 3 : t >= 3 ? 2 : t >= 1 ? 1 : 0; }

// Where the parts of the scratch begin (floats); every part a multiple of 64 floats.
struct Parts {
  int64_t starts, totals, u, w, kt, end;
};
__host__ __device__ inline int64_t padded_rows(int N) { return N <= 32 ? 32 : N <= 64 ? 64 : N <= 128 ? 128 : 256; }
__host__ __device__ inline Parts parts_of(int num_chunks, int heads, int N, int P, int delta) {
  const int64_t units = (int64_t)num_chunks * heads;
  const int64_t np = padded_rows(N);
  const int64_t pp = (P + 15) / 16 * 16;
  Parts p;
  p.starts = 0;                                            // S in front of a chunk, [PT][NT][64][4]
  p.totals = p.starts + units * np * pp;                   // the chunk's whole decay, [np]
  p.u = p.totals + units * np;                             // Y, then u: [PT][4][64][4]
  p.w = p.u + (delta ? units * kTok * pp : 0);             // -W: [4][NT][64][4]
  p.kt = p.w + (delta ? units * kTok * np : 0);            // decayed keys: [NT][4][64][4]
  p.end = p.kt + (delta ? units * kTok * np : 0);
  return p;
}

// The same for linear forms in two launches.
struct ScanParts {
  int64_t q, k, p, d0, scale, whole, end;
};
__host__ __device__ inline ScanParts scan_parts_of(int num_chunks, int heads, int kv_heads, int N) {
  const int64_t units = (int64_t)num_chunks * heads, shared = (int64_t)num_chunks * kv_heads;
  ScanParts p;
  p.q = 0;                                                 // [4][NT][64][4]
  p.k = p.q + shared * kTok * padded_rows(N);              // [NT][4][64][4]
  p.p = p.k + shared * kTok * padded_rows(N);              // (q . k) M vs: [10][64][4]
  p.d0 = p.p + units * kTiles * 256;                       // D(t), [64]
  p.scale = p.d0 + units * kTok;                           // M(last, s) vs, [64]
  p.whole = p.scale + units * kTok;                        // M(last, first) times the first's own
  p.end = p.whole + units;
  return p;
}

// Rows [first, first + nt) of x, N columns from `col`, into dst [64][NP + 4]; zeros elsewhere.
// SiLU, or the rotation of neighbours by a token's row of the table and a factor, on the way.
// A thread takes the same four columns of every 256 / (NP / 4)-th row, all asked for at once.
template <int NP, int FORM>
__device__ __forceinline__ void stage_rows(const ChunkedArgs& a, float* dst, int col, int first,
                                           int nt, int pos0, bool key, bool wide) {
  constexpr int Q = NP / 4, STEP = kThreads / Q, COUNT = kTok / STEP;
  const int t0 = threadIdx.x / Q, n = threadIdx.x % Q * 4, left = a.N - n;
  const float* row = a.x + (int64_t)first * a.ld + col + n;
  auto put = [&](int t, f32x4 v) {
    if (FORM == kSilu) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = silu(v[j]);
    }
    if (FORM == kTurned) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (n + 2 * j < a.turn_dims) {                 // (rows behind the last are zeros)
          const float2 c = a.turn[(int64_t)(pos0 + min(t, nt - 1)) * (a.turn_dims / 2) + n / 2 + j];
          const float even = v[2 * j], odd = v[2 * j + 1];
          v[2 * j] = fmaf(odd, -c.y, even * c.x);
          v[2 * j + 1] = fmaf(even, c.y, odd * c.x);
        }
      }
      if (key) v *= a.k_scale;
    }
    write4(dst + t * (NP + 4) + n, v);
    if (FORM == kTurned) __builtin_amdgcn_sched_barrier(0);      // (or every angle is asked for at once)
  };
  if (wide) {
    // (no load under a condition of its own: the compiler waits inside it, and what was to be asked for
    // at once was a trip to memory after the other)
    const float* from = left > 0 ? row : row - n;
    f32x4 v[COUNT];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) v[u] = read4(from + (int64_t)min(t0 + u * STEP, nt - 1) * a.ld);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const int t = t0 + u * STEP;
      put(t, t < nt && left > 0 ? v[u] : f32x4{0.f, 0.f, 0.f, 0.f});
    }
  } else {
#pragma unroll 2
    for (int u = 0; u < COUNT; ++u) {
      const int t = t0 + u * STEP;
      const float* from = row - n + (int64_t)min(t, nt - 1) * a.ld;
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = from[min(n + j, a.N - 1)];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = t < nt && left > j ? v[j] : 0.f;
      put(t, v);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// Decays per row of S, gates rows of head h, into dst [64][NP + 4]; ones elsewhere.
template <int NP>
__device__ __forceinline__ void stage_decays(const ChunkedArgs& a, float* dst, int h, int first, int nt) {
  constexpr int COUNT = kTok * NP / kThreads, AT_ONCE = COUNT < 16 ? COUNT : 16;
  static_assert(kTok * NP % kThreads == 0 && COUNT % AT_ONCE == 0, "whole turns");
  const float* from = a.gates + (int64_t)first * a.ldg + a.heads + h * a.N;
#pragma unroll 1
  for (int u0 = 0; u0 < COUNT; u0 += AT_ONCE) {
    float v[AT_ONCE];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      const int i = threadIdx.x + (u0 + u) * kThreads;
      v[u] = from[(int64_t)min(i / NP, nt - 1) * a.ldg + min(i % NP, a.N - 1)];
    }
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      const int i = threadIdx.x + (u0 + u) * kThreads, t = i / NP, n = i % NP;
      dst[t * (NP + 4) + n] = t < nt && n < a.N ? v[u] : 1.f;
    }
  }
}

// Token t's decay of head h (one for all rows) and the factor on its v.
__device__ __forceinline__ void token_scalars(const ChunkedArgs& a, int t, int h, float& g, float& vs) {
  vs = 1.f;
  if (a.dt) {
    vs = softplus(a.dt[(int64_t)t * a.ldg + h] + a.dt_bias[h]);
    g = expf(-expf(a.a_log[h]) * vs);
  } else {
    g = a.gates ? (a.per_row ? 1.f : a.gates[(int64_t)t * a.ldg + a.heads + h]) : a.decay[h];
  }
}

// A head's decays in a chunk, in LDS.  M(t, s) between blocks of 16 tokens is pre[t] (the decays
// from t's block's first token through t) times the whole decays of the blocks between times
// suf[s] (those behind s in its block).
struct HeadDecays {
  static constexpr int kFloats = 6 * kTok + 4;
  float* at;
  __device__ float* g() const { return at; }
  __device__ float* pre() const { return at + kTok; }
  __device__ float* suf() const { return at + 2 * kTok; }
  __device__ float* d0() const { return at + 3 * kTok; }      // D(t)
  __device__ float* es() const { return at + 4 * kTok; }      // M(last, s)
  __device__ float* vs() const { return at + 5 * kTok; }
  __device__ float* total() const { return at + 6 * kTok; }   // of the four blocks
};

// One wavefront, a token a lane (dec 1 behind the chunk's end), fills them in.  The products are
// made by doubling, in 64 bits: equal decays have equal roundings, which every doubling doubles (a
// chunk's whole decay was off by up to 32 of them, and every chunk's by the same: with decays of
// 1 - 2^-9 outputs by 1.7e-6 instead of 4.6e-7).
__device__ __forceinline__ void spread_decays(HeadDecays d, float dec, float vs, int lane) {
  const int l = lane % 16, blk = lane / 16;
  double p = dec, q = dec;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const double x = __shfl_up(p, o, 16), y = __shfl_down(q, o, 16);
    p *= l >= o ? x : 1.;
    q *= l + o < 16 ? y : 1.;
  }
  const double behind = __shfl_down(q, 1, 16), suf = l < 15 ? behind : 1.;
  const double t0 = __shfl(p, 15, 64), t1 = __shfl(p, 31, 64), t2 = __shfl(p, 47, 64), t3 = __shfl(p, 63, 64);
  d.g()[lane] = dec;
  d.pre()[lane] = (float)p;
  d.suf()[lane] = (float)suf;
  d.vs()[lane] = vs;
  d.d0()[lane] = (float)(p * (blk == 0 ? 1. : blk == 1 ? t0 : blk == 2 ? t0 * t1 : t0 * t1 * t2));
  d.es()[lane] = (float)(suf * (blk == 3 ? 1. : blk == 2 ? t3 : blk == 1 ? t2 * t3 : t1 * t2 * t3));
  if (l == 15) d.total()[blk] = (float)p;
}

// One wavefront, a token of a chunk a lane (dec 1 behind its end): M(last, token), and the chunk's whole
// decay in lane 0.  Products by doubling, in 64 bits, as above.
__device__ __forceinline__ float decay_behind(float dec, int lane, float& whole) {
  double p = dec;                          // from this token through the last
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double q = __shfl_down(p, o, 64);
    p *= lane + o < 64 ? q : 1.;
  }
  const double behind = __shfl_down(p, 1, 64);
  whole = (float)p;
  return (float)(lane < 63 ? behind : 1.);
}

// M(t, s) times vs(s) for rows t = 4 g + r and column s = l of tile (i, j), j <= i; zero above the
// diagonal.  Multiplied up in 64 bits and rounded once.
__device__ __forceinline__ f32x4 tile_decays(HeadDecays d, int i, int j, int l, int g) {
  f32x4 m;
  const double vs = d.vs()[16 * j + l];
  if (i == j) {
    const float* gb = d.g() + 16 * i;
    double run = 1.;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      run = u > l ? run * gb[u] : 1.;
      if (u / 4 == g) m[u % 4] = u >= l ? (float)(run * vs) : 0.f;
    }
    return m;
  }
  double col = d.suf()[16 * j + l] * vs;
  for (int b = j + 1; b < i; ++b) col *= d.total()[b];
  const f32x4 row = read4(d.pre() + 16 * i + 4 * g);
#pragma unroll
  for (int r = 0; r < 4; ++r) m[r] = (float)(row[r] * col);
  return m;
}

// One 16 x 16 tile of rows a . rows b over NP columns, both in LDS.
template <int NT>
__device__ __forceinline__ f32x4 gram_tile(const float* a, const float* b, int l, int g) {
  constexpr int LD = 16 * NT + 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto part = [&](int j) {
    return product4(read4(a + l * LD + 16 * j + 4 * g), read4(b + l * LD + 16 * j + 4 * g));
  };
#pragma unroll 2
  for (int j = 0; j < NT; j += 2) acc += part(j) + part(j + 1);
  return acc;
}

// The sum over the sixteen lanes of a row, in every one of them.
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int step = 0; step < 4; ++step) {
    const int x = __builtin_bit_cast(int, v);
    const int y = step == 0   ? __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true)     // neighbour
                  : step == 1 ? __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true)     // of the quad
                  : step == 2 ? __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true)    // mirrored eight
                              : __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true);   // turned by eight
    v += __builtin_bit_cast(float, y);
  }
  return v;
}

template <int PER>
__device__ __forceinline__ void read_run(const float* p, float (&v)[PER]) {
  if constexpr (PER % 4 == 0) {
#pragma unroll
    for (int j = 0; j < PER / 4; ++j) {
      const f32x4 x = read4(p + 4 * j);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[4 * j + r] = x[r];
    }
  } else {
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = p[j];
  }
}

// T u for a diagonal tile T (its left operand), zero above its diagonal: row t takes u of its own and of
// earlier tokens.  Zero times what is not finite is not zero, so where such u are among the
// sixteen a row at a time is made, with the later ones left out, and taken.
__device__ __forceinline__ f32x4 causal_product(f32x4 a, f32x4 u, int g) {
  if (__builtin_amdgcn_ballot_w64(!(fabsf(u[0]) + fabsf(u[1]) + fabsf(u[2]) + fabsf(u[3]) < INFINITY)) == 0)
    return product4(a, u);
  f32x4 out;
#pragma unroll 1
  for (int t = 0; t < 16; ++t) {
    f32x4 seen;
#pragma unroll
    for (int r = 0; r < 4; ++r) seen[r] = 4 * g + r <= t ? u[r] : 0.f;
    const f32x4 sums = product4(a, seen);
#pragma unroll
    for (int r = 0; r < 4; ++r) out[r] = 4 * g + r == t ? sums[r] : out[r];
  }
  return out;
}

// Decays per row: the diagonal tiles (wavefront w takes block w), the products' decays
// multiplied up pair by pair.  left: q or k rows.  STRICT leaves the diagonal out.  Sixteen lanes
// share a column s (a run of channels each), four columns at a time.
template <int NP, bool STRICT>
__device__ __forceinline__ void diagonal_tiles(float* tiles, const float* left, const float* k,
                                               const float* gr, int w, int lane) {
  constexpr int LD = NP + 4, PER = NP / 16;
  const int n0 = lane % 16 * PER;
  float* tile = tiles + tri(w, w) * kTile;
  for (int s0 = 0; s0 < 16; s0 += 4) {
    const int s = s0 + lane / 16;
    float kw[PER], mine = 0.f;              // the lane with l = t keeps row t
    read_run<PER>(k + (16 * w + s) * LD + n0, kw);
    for (int t = s0; t < 16; ++t) {
      float x[PER], d[PER], part = 0.f;
      read_run<PER>(left + (16 * w + t) * LD + n0, x);
      read_run<PER>(gr + (16 * w + t) * LD + n0, d);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        kw[j] *= t > s ? d[j] : 1.f;
        part = fmaf(x[j], kw[j], part);
      }
      part = row_sum(part);
      if (lane % 16 == t) mine = t > s || (t == s && !STRICT) ? part : 0.f;
    }
    tile[lane % 16 * kTileLd + s] = mine;
  }
}

// Decays per row, in place, a (block, channel) a thread: `pre` rows times the decays from their
// block's first token through their own, `post` rows (into gr) times those behind their own in
// the block, and a block's whole decay into blocks [4][NP].
template <int NP>
__device__ __forceinline__ void split_decays(float* pre, const float* post, float* gr, float* blocks) {
  constexpr int LD = NP + 4;
  for (int i = threadIdx.x; i < 4 * NP; i += kThreads) {
    const int blk = i / NP, n = i % NP;
    float g[16], k[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      g[t] = gr[(16 * blk + t) * LD + n];
      k[t] = post[(16 * blk + t) * LD + n];
    }
    double m = 1.;                         // (rounded where it is used, not at every step)
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      m *= g[t];
      pre[(16 * blk + t) * LD + n] = (float)(pre[(16 * blk + t) * LD + n] * m);
    }
    blocks[i] = (float)m;
    m = 1.;
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      gr[(16 * blk + t) * LD + n] = (float)(k[t] * m);
      m *= g[t];
    }
  }
}

// The tile (i, j), j < i, of the products with decays per row: pre rows of block i, post rows of
// block j, and the whole decays of the blocks between.
template <int NT>
__device__ __forceinline__ f32x4 split_tile(const float* pre, const float* post, const float* blocks,
                                            int i, int j, int l, int g) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto part = [&](int c) {
    const int n = 16 * c + 4 * g;
    f32x4 b = read4(post + (16 * j + l) * LD + n);
    for (int m = j + 1; m < i; ++m) b *= read4(blocks + m * NP + n);
    return product4(read4(pre + (16 * i + l) * LD + n), b);
  };
#pragma unroll 2
  for (int c = 0; c < NT; c += 2) acc += part(c) + part(c + 1);
  return acc;
}

// `tiles`: of 16 tokens that are worked on.  One, for the single tokens that decode beside a
// prompt, or all four (rows behind the chunk's end are zeros): so that the loops over them unroll.
struct ChunkRange {
  int first, nt, entry, tiles, pos0;
};
__device__ __forceinline__ int chunk_tiles(int nt) { return nt <= 16 ? 1 : 4; }
__device__ __forceinline__ ChunkRange chunk_range(const ChunkedArgs& a, int chunk) {
  ChunkRange c;
  c.first = a.chunks[3 * chunk];
  c.nt = a.chunks[3 * chunk + 1] - c.first;
  c.entry = a.chunks[3 * chunk + 2];
  c.tiles = chunk_tiles(c.nt);
  c.pos0 = a.b.positions[c.first];
  return c;
}

// ---------------------------------------------------------------- linear forms: a chunk's own share
// A workgroup takes one chunk and `heads_each` (up to 8) heads that read the same keys; 64
// columns of v at a time lie in LDS, scaled by M(last, s) vs_s, the next 64 on their way.
template <int NT, int FORM>
__global__ __launch_bounds__(kThreads, 2) void chunk_local_kernel(ChunkedArgs a, int heads_each, int wide) {
  constexpr int NP = 16 * NT, LD = NP + 4, VC = 64, LV = VC + 4, OWN = (NT + 3) / 4;
  constexpr int EACH = kTok * VC / kThreads;
  extern __shared__ __align__(16) float lds[];
  float* Ks = lds;
  float* Vs = Ks + kTok * LD;
  float* scale = Vs + kTok * LV;          // [heads_each][64]
  const int chunk = blockIdx.y, h0 = blockIdx.x * heads_each;
  const ChunkRange c = chunk_range(a, chunk);
  const int hk = h0 / (a.heads / a.kv_heads), PT = (a.P + 15) / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const Parts parts = parts_of(a.num_chunks, a.heads, a.N, a.P, 0);
  const int vt = threadIdx.x / VC, vp = threadIdx.x % VC;       // a thread's first token, its column
  float v[EACH];
  auto fetch = [&](int h, int c0) {
    const float* col = a.x + a.v_col + h * a.P + c0 + vp;
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
      const int t = vt + u * (kThreads / VC);
      v[u] = t < c.nt && c0 + vp < a.P ? col[(int64_t)(c.first + t) * a.ld] : 0.f;
    }
  };
  fetch(h0, 0);
  for (int i = w; i < heads_each; i += 4) {
    float dec = 1.f, vs = 0.f;
    if (lane < c.nt) token_scalars(a, c.first + lane, h0 + i, dec, vs);
    float whole;
    scale[i * kTok + lane] = vs * decay_behind(dec, lane, whole);
    if (lane == 0) a.scratch[parts.totals + ((int64_t)chunk * a.heads + h0 + i) * NP] = whole;
  }
  stage_rows<NP, FORM>(a, Ks, a.k_col + hk * a.N, c.first, c.nt, c.pos0, true, wide);
  __syncthreads();
  f32x4 kf[OWN][4];
#pragma unroll
  for (int o = 0; o < OWN; ++o)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * (w + 4 * o) + l;
        kf[o][j][r] = n < NP ? Ks[(16 * j + 4 * g + r) * LD + n] : 0.f;
      }
  for (int i = 0; i < heads_each; ++i) {
    const int h = h0 + i;
    float* share = a.scratch + parts.starts + ((int64_t)chunk * a.heads + h) * PT * NT * 256;
    for (int c0 = 0; c0 < a.P; c0 += VC) {
      __syncthreads();                     // the columns before have been read
#pragma unroll
      for (int u = 0; u < EACH; ++u) {
        const int t = vt + u * (kThreads / VC);
        Vs[t * LV + vp] = (FORM == kSilu ? silu(v[u]) : v[u]) * scale[i * kTok + t];
      }
      if (c0 + VC < a.P) fetch(h, c0 + VC);
      else if (i + 1 < heads_each) fetch(h + 1, 0);
      __syncthreads();
      for (int ct = 0; ct < VC / 16 && c0 / 16 + ct < PT; ++ct) {
        f32x4 vf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) vf[j][r] = Vs[(16 * j + 4 * g + r) * LV + 16 * ct + l];
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
          if (w + 4 * o >= NT) break;
          const f32x4 early = product2(kf[o][0], vf[0]) + product2(kf[o][1], vf[1]);
          const f32x4 acc = early + (product2(kf[o][2], vf[2]) + product2(kf[o][3], vf[3]));
          write4(share + ((int64_t)(c0 / 16 + ct) * NT + w + 4 * o) * 256 + lane * 4, acc);
        }
      }
    }
  }
}

// The chunks of an entry in order, four elements of S a thread: the scratch holds a chunk's own
// share and receives the state in front of the chunk.
template <int NT>
__global__ __launch_bounds__(kThreads) void chunk_carry_kernel(ChunkedArgs a) {
  const int h = blockIdx.x, e = blockIdx.y, PT = (a.P + 15) / 16;
  const int i = blockIdx.z * kThreads + threadIdx.x;
  if (i >= PT * NT * 64) return;
  const int lane = i % 64, l = lane % 16, g = lane / 16;
  const int n0 = i / 64 % NT * 16 + 4 * g, p = i / 64 / NT * 16 + l;
  const Parts parts = parts_of(a.num_chunks, a.heads, a.N, a.P, 0);
  float* st = a.state + ((int64_t)a.b.slot_ids[e] * a.heads + h) * a.N * a.P;
  const bool fresh = a.b.positions[a.b.q_start[e]] == 0;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (!fresh && n0 + r < a.N && p < a.P) S[r] = st[(int64_t)(n0 + r) * a.P + p];
  const int64_t stride = (int64_t)a.heads * PT * NT * 256;
  const int begin = a.entry_chunks[e], end = a.entry_chunks[e + 1];
  float* at = a.scratch + parts.starts + begin * stride + (int64_t)h * PT * NT * 256 + (int64_t)i * 4;
  const float* total = a.scratch + parts.totals + ((int64_t)begin * a.heads + h) * NT * 16;
  constexpr int AHEAD = 4;                 // shares on their way
  f32x4 next[AHEAD];
  float dec[AHEAD];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    if (begin + u < end) {
      next[u] = read4(at + u * stride);
      dec[u] = total[(int64_t)u * a.heads * NT * 16];
    }
  }
  for (int c = begin; c < end; c += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (c + u >= end) break;
      const f32x4 share = next[u];
      const float d = dec[u];
      if (c + u + AHEAD < end) {
        next[u] = read4(at + (int64_t)(c + u + AHEAD - begin) * stride);
        dec[u] = total[(int64_t)(c + u + AHEAD - begin) * a.heads * NT * 16];
      }
      write4(at + (int64_t)(c + u - begin) * stride, S);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] = fmaf(d, S[r], share[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n0 + r < a.N && p < a.P) st[(int64_t)(n0 + r) * a.P + p] = S[r];
}

// ---------------------------------------------------------------- linear forms in two launches
// Three launches write the state in front of every chunk, add them up and read them again (at 64 heads
// of 128 x 64 and 2,048 tokens 270 MB of their 123 us).  Here one makes what does not hang on the
// state, in the order in which the matrix cores take it: q, k, and (q . k) times the decays; the other
// walks, with the state in registers, and nothing of it is written but the last.
// A workgroup of the first takes one chunk and `heads_each` (up to 8) heads that read the same q and k.
// Decays are multiplied up in the order that the three launches have, and every sum is theirs: the bits
// are the same.  (In an order of this form's own the first took 28.5 us instead of 29.5 at that size;
// with the tiles dealt out in turn, two of the diagonal to one wavefront, 32.5.)
template <int NT, int FORM, int RT>
__device__ __forceinline__ void prepare_chunk(const ChunkedArgs& a, const ChunkRange& c, int heads_each,
                                              int wide) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  extern __shared__ __align__(16) float lds[];
  float* Qs = lds;
  float* Ks = Qs + kTok * LD;
  float* decays = Ks + kTok * LD;         // [heads_each] of HeadDecays
  const int chunk = blockIdx.y, h0 = blockIdx.x * heads_each;
  const int group = a.heads / a.kv_heads, hk = h0 / group;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const ScanParts parts = scan_parts_of(a.num_chunks, a.heads, a.kv_heads, a.N);
  float dec[2] = {1.f, 1.f}, vs[2] = {0.f, 0.f};          // of heads w and w + 4, a token a lane
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (w + 4 * u < heads_each && lane < c.nt)
      token_scalars(a, c.first + lane, h0 + w + 4 * u, dec[u], vs[u]);
  stage_rows<NP, FORM>(a, Qs, a.q_col + hk * a.N, c.first, c.nt, c.pos0, false, wide);
  stage_rows<NP, FORM>(a, Ks, a.k_col + hk * a.N, c.first, c.nt, c.pos0, true, wide);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (w + 4 * u < heads_each) {
      const HeadDecays d{decays + (w + 4 * u) * HeadDecays::kFloats};
      spread_decays(d, dec[u], vs[u], lane);
      const int64_t unit = (int64_t)chunk * a.heads + h0 + w + 4 * u;
      a.scratch[parts.d0 + unit * kTok + lane] = d.d0()[lane];
      float whole;
      a.scratch[parts.scale + unit * kTok + lane] = vs[u] * decay_behind(dec[u], lane, whole);
      if (lane == 0) a.scratch[parts.whole + unit] = whole;
    }
  }
  __syncthreads();
  // A wavefront's tiles: one on the diagonal, whose decays take longest, one or two below it (row 4 or
  // more: none).
  auto tile_row = [&](int u) { return u == 0 ? w : u == 1 ? min(w + 1, 3) : w < 2 ? w + 2 : 4; };
  auto tile_col = [&](int u) { return u == 0 ? w : u == 1 ? (w < 2 ? w : w - 1) : 0; };
  f32x4 gram[3];
#pragma unroll
  for (int u = 0; u < 3; ++u)
    if (tile_row(u) < RT) gram[u] = gram_tile<NT>(Qs + 16 * tile_row(u) * LD, Ks + 16 * tile_col(u) * LD, l, g);
  if (h0 % group == 0) {                  // q and k themselves, by the first workgroup that reads them
    const int64_t unit = (int64_t)chunk * a.kv_heads + hk;
    if (w < RT) {
      float* to = a.scratch + parts.q + (unit * 4 + w) * NT * 256 + lane * 4;
#pragma unroll
      for (int j = 0; j < NT; ++j) write4(to + j * 256, read4(Qs + (16 * w + l) * LD + 16 * j + 4 * g));
    }
    for (int n = w; n < NT; n += 4) {
      float* to = a.scratch + parts.k + (unit * NT + n) * 4 * 256 + lane * 4;
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = Ks[(16 * j + 4 * g + r) * LD + 16 * n + l];
        write4(to + j * 256, v);
      }
    }
  }
  for (int h = 0; h < heads_each; ++h) {
    const HeadDecays d{decays + h * HeadDecays::kFloats};
    // (row 4 g + r and column l of a tile go where a left operand has them: 16 bytes at a time)
    float* to = a.scratch + parts.p + ((int64_t)chunk * a.heads + h0 + h) * kTiles * 256 +
                (l / 4 * 16 + 4 * g) * 4 + l % 4;
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int i = tile_row(u), j = tile_col(u);
      if (i < RT) {
        const f32x4 m = tile_decays(d, i, j, l, g);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          to[tri(i, j) * 256 + r * 4] = i > j || 4 * g + r >= l ? gram[u][r] * m[r] : 0.f;
      }
    }
  }
}

template <int NT, int FORM>
__global__ __launch_bounds__(kThreads) void chunk_prepare_kernel(ChunkedArgs a, int heads_each, int wide) {
  const ChunkRange c = chunk_range(a, blockIdx.y);
  if (c.tiles == 1) prepare_chunk<NT, FORM, 1>(a, c, heads_each, wide);
  else prepare_chunk<NT, FORM, 4>(a, c, heads_each, wide);
}

// The chunks of an entry in order, sixteen columns of S a workgroup, with their outputs.  Of eight
// wavefronts, two to a SIMD, w = 0 to 3 keep the rows of tiles w, w + 4, ... of S and make their new
// values; a chunk's own share of S does not hang on S, so they meet the others, which make the outputs
// of 16 tokens each, once a chunk, when the state in front of it and v lie in LDS (in one of two
// buffers: whoever still reads the other is in the chunk before).  An operand of a chunk some turns
// ahead is asked for as soon as its registers have been read; nothing in the loops that touches memory
// hangs on a condition, so that a wait is for the operands it is for.
// A chunk of 128 x 16 of S takes 2.3 us: 1.2 are a SIMD's products, 1.4 the 108 loads that a unit takes
// in 28 cycles each, and neither hides the other whole (without loads 1.8, without the meetings 1.9; as
// four wavefronts that do both parts 2.6).
constexpr int kScanThreads = 512;

// Four bytes a lane, at `offset` from a base that the lanes share; offsets from `bytes` on go nowhere.
__device__ __forceinline__ void store_inside(float* base, int bytes, int offset, float v) {
  const auto to = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), to, offset, 0, 0);
}

template <int NT>
struct StateOperands {
  static constexpr int OWN = (NT + 3) / 4;
  f32x4 k[OWN][4], v, scale;
  float total;
};

template <int NT>
struct OutputOperands {
  f32x4 q[NT], p[4], d0;
};

// turn(i, c) for c = 0 to count - 1, i = c % RING known to the compiler.
template <int RING, typename F>
__device__ __forceinline__ void in_turns(int count, F turn) {
  int c = 0;
  for (; c + RING <= count; c += RING) {
#pragma unroll
    for (int i = 0; i < RING; ++i) turn(i, c + i);
  }
#pragma unroll
  for (int i = 0; i < RING - 1; ++i)
    if (c + i < count) turn(i, c + i);
}

template <int NT, int FORM>
__global__ __launch_bounds__(kScanThreads, 1) void chunk_scan_kernel(ChunkedArgs a) {
  constexpr int OWN = (NT + 3) / 4;
  __shared__ __align__(16) float s_lds[2][NT][256];
  __shared__ __align__(16) float v_lds[2][2][4][256];     // scaled, and as it stands
  // (heads that read the same q and k on one XCD: they lie next to each other, workgroups do not)
  const int h = a.heads % 8 == 0 ? (int)(blockIdx.x % 8) * (a.heads / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
  const int e = blockIdx.z, ct = blockIdx.y, hk = h / (a.heads / a.kv_heads);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), w = wave % 4;
  const int lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const int p = 16 * ct + l, first_row = 16 * w + 4 * g;
  const ScanParts parts = scan_parts_of(a.num_chunks, a.heads, a.kv_heads, a.N);
  const int q0 = a.b.q_start[e], tokens = a.b.q_start[e + 1] - q0;
  const int begin = a.entry_chunks[e], count = a.entry_chunks[e + 1] - begin;
  if (count < 1) return;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const float* v_col = a.x + a.v_col + h * a.P + min(p, a.P - 1);
  auto unit_of = [&](int c) { return (int64_t)(begin + min(c, count - 1)) * a.heads + h; };
  auto shared_of = [&](int c) { return (int64_t)(begin + min(c, count - 1)) * a.kv_heads + hk; };

  if (wave < 4) {
    float* st = a.state + ((int64_t)a.b.slot_ids[e] * a.heads + h) * a.N * a.P;
    const bool fresh = a.b.positions[q0] == 0;
    f32x4 S[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      S[o] = zero;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * (w + 4 * o) + 4 * g + r;
        if (!fresh && n < a.N && p < a.P) S[o][r] = st[(int64_t)n * a.P + p];
      }
    }
    // only the last chunk may be short; of one of a single tile nothing else was left
    const int one_tile = tokens - (count - 1) * kTok <= 16 ? count - 1 : count;
    const bool owns_last = NT % 4 == 0 || w + 4 * (OWN - 1) < NT;
    auto fetch_v = [&](StateOperands<NT>& f, int c) {
      const int64_t unit = unit_of(c);
#pragma unroll
      for (int r = 0; r < 4; ++r) f.v[r] = v_col[(int64_t)(q0 + min(c * kTok + first_row + r, tokens - 1)) * a.ld];
      f.scale = read4(a.scratch + parts.scale + unit * kTok + first_row);
      f.total = a.scratch[parts.whole + unit];
    };
    auto fetch_k = [&](StateOperands<NT>& f, int c, int o) {
      const float* at = a.scratch + parts.k + shared_of(c) * NT * 1024 + min(w + 4 * o, NT - 1) * 1024;
#pragma unroll
      for (int j = 0; j < 4; ++j) f.k[o][j] = read4(at + j * 256 + lane * 4);
    };
    auto walk = [&](auto size) {
      constexpr bool MORE = decltype(size)::value > 0;
      constexpr int RING = MORE ? decltype(size)::value : 1;
      StateOperands<NT> ring[RING];
#pragma unroll
      for (int i = 0; i < RING; ++i) {
        fetch_v(ring[i], i);
#pragma unroll
        for (int o = 0; o < OWN; ++o) fetch_k(ring[i], i, o);
      }
      in_turns<RING>(count, [&](int i, int c) {
        StateOperands<NT>& f = ring[i];
        float (&v_buf)[2][4][256] = v_lds[c & 1];
        f32x4 mine, scaled;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          mine[r] = c * kTok + first_row + r < tokens ? (FORM == kSilu ? silu(f.v[r]) : f.v[r]) : 0.f;
          scaled[r] = mine[r] * f.scale[r];
        }
        const float total = f.total;
        write4(&v_buf[0][w][lane * 4], scaled);
        write4(&v_buf[1][w][lane * 4], mine);
#pragma unroll
        for (int o = 0; o < OWN; ++o)
          if (o < OWN - 1 || owns_last) write4(&s_lds[c & 1][w + 4 * o][lane * 4], S[o]);
        __syncthreads();
        f32x4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = read4(&v_buf[0][j][lane * 4]);
        if (MORE) fetch_v(f, c + RING);
        if (c == one_tile) {
#pragma unroll
          for (int o = 0; o < OWN; ++o)
#pragma unroll
            for (int j = 1; j < 4; ++j) f.k[o][j] = zero;
        }
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
          const f32x4 early = product2(f.k[o][0], v[0]) + product2(f.k[o][1], v[1]);
          const f32x4 share = early + (product2(f.k[o][2], v[2]) + product2(f.k[o][3], v[3]));
#pragma unroll
          for (int r = 0; r < 4; ++r) S[o][r] = fmaf(total, S[o][r], share[r]);
        }
        if (MORE) {
#pragma unroll
          for (int o = 0; o < OWN; ++o) fetch_k(f, c + RING, o);
        }
      });
    };
    if (count == 1) walk(std::integral_constant<int, 0>{});
    else walk(std::integral_constant<int, 3>{});
#pragma unroll
    for (int o = 0; o < OWN; ++o)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * (w + 4 * o) + 4 * g + r;
        if (n < a.N && p < a.P) st[(int64_t)n * a.P + p] = S[o][r];
      }
    return;
  }

  const float skip = a.d_skip ? a.d_skip[h] : 0.f;
  const int out_ld = a.heads * a.P, out_at = p < a.P ? (first_row * out_ld + h * a.P + p) * 4 : -16 * out_ld;
  const float* q_at = a.scratch + parts.q + w * NT * 256 + lane * 4;
  const float* p_at = a.scratch + parts.p + tri(w, 0) * 256 + lane * 4;
  auto fetch_q = [&](OutputOperands<NT>& f, const float* at, int j) { f.q[j] = read4(at + j * 256); };
  auto fetch_p = [&](OutputOperands<NT>& f, int c) {      // (the last: the diagonal's)
    const float* at = p_at + unit_of(c) * kTiles * 256;
#pragma unroll
    for (int j = 0; j < 4; ++j) f.p[j] = read4(at + (j < 3 ? min(j, w) : w) * 256);
    f.d0 = read4(a.scratch + parts.d0 + unit_of(c) * kTok + first_row);
  };
  auto walk = [&](auto size) {
    constexpr bool MORE = decltype(size)::value > 0;
    constexpr int RING = MORE ? decltype(size)::value : 1;
    OutputOperands<NT> ring[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) {
#pragma unroll
      for (int j = 0; j < NT; ++j) fetch_q(ring[i], q_at + shared_of(i) * 4 * NT * 256, j);
      fetch_p(ring[i], i);
    }
    in_turns<RING>(count, [&](int i, int c) {
      OutputOperands<NT>& f = ring[i];
      const float* later = q_at + shared_of(c + RING) * 4 * NT * 256;
      __syncthreads();
      f32x4 s[NT], v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = read4(&v_lds[c & 1][1][j < 3 ? j : w][lane * 4]);
#pragma unroll
      for (int j = 0; j < NT; ++j) s[j] = read4(&s_lds[c & 1][j][lane * 4]);
      // (products of earlier tokens with tiles that are not there count nothing, whatever v is)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = j < w ? v[j][r] : 0.f;
      const f32x4 x0 = product2(f.p[0], v[0]), x1 = product2(f.p[1], v[1]), x2 = product2(f.p[2], v[2]);
      const f32x4 own = causal_product(f.p[3], v[3], g);
      f32x4 acc = zero;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        acc += product2(f.q[j], s[j]);
        asm volatile("" : "+v"(acc));        // (left alone, every sum is put off to the end)
        if (MORE) fetch_q(f, later, j);
      }
      acc *= f.d0;
      acc += w == 1 ? x0 + own : w == 0 ? own : x0 + x1;
      if (w > 1) acc += w == 2 ? own : x2 + own;
      if (MORE) fetch_p(f, c + RING);
      const int nt = min(tokens - c * kTok, kTok);
      float* out = a.out + (int64_t)(q0 + c * kTok) * out_ld;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        store_inside(out, nt * out_ld * 4, out_at + r * out_ld * 4, fmaf(skip, v[3][r], acc[r]));
    });
  };
  if (count == 1) walk(std::integral_constant<int, 0>{});
  else walk(std::integral_constant<int, NT <= 4 ? 3 : 2>{});
}

// ---------------------------------------------------------------- delta rule: Y, W, decayed keys
// A workgroup takes one chunk of one head: the 64 x 64 triangular matrix in LDS, its diagonal
// blocks inverted (a wavefront each, a column a lane), then block by block the solution for the
// columns of W and Y, 16 columns of a right side at a time in a wavefront's registers.
template <int NT, bool ROW, int RT>
__device__ __forceinline__ void solve_chunk(const ChunkedArgs& a, const ChunkRange& c, int wide) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  extern __shared__ __align__(16) float lds[];
  float* Ks = lds;
  float* Gs = Ks + kTok * LD;                             // ROW only
  float* tiles = Gs + (ROW ? kTok * LD : 0);
  float* beta = tiles + kTiles * kTile;
  const HeadDecays dec{beta + kTok};
  float* blocks = dec.at;                                 // ROW only: [4][NP]
  const int chunk = blockIdx.y, h = blockIdx.x;
  const int hk = h / (a.heads / a.kv_heads), PT = (a.P + 15) / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const int64_t unit = (int64_t)chunk * a.heads + h;
  const Parts parts = parts_of(a.num_chunks, a.heads, a.N, a.P, 1);
  stage_rows<NP, kPlain>(a, Ks, a.k_col + hk * a.N, c.first, c.nt, c.pos0, true, wide);
  if (ROW) stage_decays<NP>(a, Gs, h, c.first, c.nt);
  if (threadIdx.x < kTok) {
    float g1 = 1.f, vs = 1.f;
    if (lane < c.nt) token_scalars(a, c.first + lane, h, g1, vs);
    beta[lane] = lane < c.nt ? a.gates[(int64_t)(c.first + lane) * a.ldg + h] : 0.f;
    if (!ROW) spread_decays(dec, g1, vs, lane);
  }
  __syncthreads();
  // minus the matrix below its diagonal
  if (ROW) {
    if (w < RT) diagonal_tiles<NP, true>(tiles, Ks, Ks, Gs, w, lane);
    __syncthreads();
    split_decays<NP>(Ks, Ks, Gs, blocks);     // Ks: decayed to, Gs: decayed from
    __syncthreads();
    for (int t = w; t < kTiles; t += 4) {
      const int i = tri_row(t), j = t - tri(i, 0);
      if (i >= RT) break;
      f32x4 acc;
      if (i == j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = tiles[t * kTile + (4 * g + r) * kTileLd + l];
      } else {
        acc = split_tile<NT>(Ks, Gs, blocks, i, j, l, g);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        tiles[t * kTile + (4 * g + r) * kTileLd + l] = -beta[16 * i + 4 * g + r] * acc[r];
    }
  } else {
    for (int t = w; t < kTiles; t += 4) {
      const int i = tri_row(t), j = t - tri(i, 0);
      if (i >= RT) break;
      f32x4 m = gram_tile<NT>(Ks + 16 * i * LD, Ks + 16 * j * LD, l, g) * tile_decays(dec, i, j, l, g);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        tiles[t * kTile + (4 * g + r) * kTileLd + l] =
            i > j || 4 * g + r > l ? -beta[16 * i + 4 * g + r] * m[r] : 0.f;
    }
  }
  __syncthreads();
  // the inverse of a diagonal block: column l in lane l
  float inv[16];
  if (w < RT) {
    const float* tile = tiles + tri(w, w) * kTile;
#pragma unroll
    for (int i = 0; i < 16; ++i) inv[i] = i == l ? 1.f : 0.f;
#pragma unroll
    for (int m = 0; m < 15; ++m) {         // column m of the block times row m of the inverse
#pragma unroll
      for (int i = m + 1; i < 16; ++i) inv[i] = fmaf(tile[i * kTileLd + m], inv[m], inv[i]);
      if (m % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  if (w < RT && g == 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) tiles[tri(w, w) * kTile + i * kTileLd + l] = inv[i];
  }
  __syncthreads();
  float* W = a.scratch + parts.w + unit * kTok * NP;
  float* Y = a.scratch + parts.u + unit * PT * 4 * 256;
  for (int ct = w; ct < NT + PT; ct += 4) {
    f32x4 X[4];
    const int n = 16 * ct + l, p = n - NP;
    float whole = 1.f;                     // ROW: the decay of the blocks in front
    float vx[RT][4];                       // a column of v, all of it asked for at once
    if (ct >= NT) {
      const float* from = a.x + (int64_t)c.first * a.ld + a.v_col + h * a.P + min(p, a.P - 1);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) vx[i][r] = from[(int64_t)min(16 * i + 4 * g + r, c.nt - 1) * a.ld];
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      f32x4 acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * i + 4 * g + r;
        float v;
        if (ct < NT) v = ROW ? Ks[t * LD + n] * whole : Ks[t * LD + n] * dec.d0()[t];
        else v = t < c.nt && p < a.P ? vx[i][r] : 0.f;
        acc[r] = beta[t] * v;
      }
      if (ROW && ct < NT) whole *= blocks[i * NP + n];
#pragma unroll
      for (int m = 0; m < i; ++m)
        acc += product4(read4(tiles + tri(i, m) * kTile + l * kTileLd + 4 * g), X[m]);
      X[i] = causal_product(read4(tiles + tri(i, i) * kTile + l * kTileLd + 4 * g), acc, g);
      if (ct < NT) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          W[((i * NT + ct) * 64 + l / 4 * 16 + 4 * g + r) * 4 + l % 4] = -X[i][r];
      } else {
        write4(Y + ((ct - NT) * 4 + i) * 256 + lane * 4, X[i]);
      }
    }
  }
  float* KT = a.scratch + parts.kt + unit * kTok * NP;
  for (int nt = w; nt < NT; nt += 4) {
    const int n = 16 * nt + l;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      float behind = 1.f;
      if (ROW)
        for (int m = j + 1; m < 4; ++m) behind *= blocks[m * NP + n];
      f32x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = 16 * j + 4 * g + r;
        v[r] = ROW ? Gs[s * LD + n] * behind : Ks[s * LD + n] * dec.es()[s];
      }
      write4(KT + (nt * 4 + j) * 256 + lane * 4, v);
    }
  }
  for (int n = threadIdx.x; n < NP; n += kThreads) {
    a.scratch[parts.totals + unit * NP + n] =
        ROW ? blocks[n] * blocks[NP + n] * blocks[2 * NP + n] * blocks[3 * NP + n] : dec.d0()[kTok - 1];
  }
}

template <int NT, bool ROW>
__global__ __launch_bounds__(kThreads) void chunk_solve_kernel(ChunkedArgs a, int wide) {
  const ChunkRange c = chunk_range(a, blockIdx.y);
  if (c.tiles == 1) solve_chunk<NT, ROW, 1>(a, c, wide);
  else solve_chunk<NT, ROW, 4>(a, c, wide);
}

// The chunks of an entry in order, sixteen columns of S a workgroup.  Wavefront w keeps the rows
// of tiles w, w + 4, ... as sums' registers, which are operands of W S as they are: it shows them
// to the others through LDS, makes 16 tokens of u from all of them, and, when all have shown
// their u, multiplies its rows' decayed keys with it.  A turn is two products of a microsecond's
// length or less, a trip to memory for operands that another XCD wrote about two, so the
// operands of the next three chunks are on their way meanwhile (a ring of four in registers; one
// wavefront a SIMD).
template <int NT>
struct WalkOperands {
  static constexpr int OWN = (NT + 3) / 4;
  f32x4 w[NT], kt[OWN][4], dec[OWN], y;
};

template <int NT>
__global__ __launch_bounds__(kThreads, 1) void chunk_walk_kernel(ChunkedArgs a) {
  constexpr int NP = 16 * NT, OWN = (NT + 3) / 4;
  __shared__ __align__(16) float s_lds[NT][256];
  __shared__ __align__(16) float u_lds[4][256];
  const int h = blockIdx.x, e = blockIdx.y, ct = blockIdx.z, PT = (a.P + 15) / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const int p = 16 * ct + l;
  const Parts parts = parts_of(a.num_chunks, a.heads, a.N, a.P, 1);
  float* st = a.state + ((int64_t)a.b.slot_ids[e] * a.heads + h) * a.N * a.P;
  const bool fresh = a.b.positions[a.b.q_start[e]] == 0;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 S[OWN];
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    S[o] = zero;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * (w + 4 * o) + 4 * g + r;
      if (!fresh && n < a.N && p < a.P) S[o][r] = st[(int64_t)n * a.P + p];
    }
  }
  const int begin = a.entry_chunks[e], end = a.entry_chunks[e + 1];
  // only the last chunk may be short; one of a single tile left nothing for the other three
  const int rest = a.b.q_start[e + 1] - a.b.q_start[e] - (end - 1 - begin) * kTok;
  const int one_tile = rest <= 16 ? end - 1 : end;
  auto owns = [&](int o) { return NT % 4 == 0 || w + 4 * o < NT; };
  // (the operands are asked for a few at a time between products, where a wavefront would
  // otherwise wait for the unit to take all of them at once)
  auto unit_of = [&](int chunk) { return (int64_t)min(chunk, end - 1) * a.heads + h; };
  auto fetch_w = [&](WalkOperands<NT>& f, int64_t unit, int j) {
    f.w[j] = read4(a.scratch + parts.w + unit * kTok * NP + (w * NT + j) * 256 + lane * 4);
    if (j == 0)
      f.y = read4(a.scratch + parts.u + ((unit * PT + ct) * 4 + w) * 256 + lane * 4);
  };
  auto fetch_kt = [&](WalkOperands<NT>& f, int64_t unit, int i) {
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      if (owns(o)) {
        f.kt[o][i] = read4(a.scratch + parts.kt + unit * kTok * NP + ((w + 4 * o) * 4 + i) * 256 + lane * 4);
        if (i == 0) f.dec[o] = read4(a.scratch + parts.totals + unit * NP + 16 * (w + 4 * o) + 4 * g);
      }
    }
  };
  auto turn = [&](WalkOperands<NT>& f, WalkOperands<NT>& ahead, int chunk) {
    const int64_t unit = (int64_t)chunk * a.heads + h, later = unit_of(chunk + 3);
    float* start = a.scratch + parts.starts + (unit * PT + ct) * NT * 256 + lane * 4;
    if (chunk == one_tile) {
      if (w > 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) f.w[j] = zero;
        f.y = zero;
      }
#pragma unroll
      for (int o = 0; o < OWN; ++o)
#pragma unroll
        for (int i = 1; i < 4; ++i) f.kt[o][i] = zero;
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o)
      if (owns(o)) write4(&s_lds[w + 4 * o][lane * 4], S[o]);
    __syncthreads();
    f32x4 mine = f.y, part[2][2], s[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) s[j] = read4(&s_lds[j][lane * 4]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) product_step(part[j & 1], f.w[j], s[j], r);
      if (j > 0) mine += part[(j - 1) & 1][0] + part[(j - 1) & 1][1];
      fetch_w(ahead, later, j);
      __builtin_amdgcn_sched_barrier(0);
    }
    mine += part[(NT - 1) & 1][0] + part[(NT - 1) & 1][1];
    write4(&u_lds[w][lane * 4], mine);
    __syncthreads();
    f32x4 u[4], more[2][OWN][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = read4(&u_lds[i][lane * 4]);
    write4(a.scratch + parts.u + ((unit * PT + ct) * 4 + w) * 256 + lane * 4, mine);
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      if (owns(o)) write4(start + (w + 4 * o) * 256, S[o]);
      S[o] *= f.dec[o];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int o = 0; o < OWN; ++o)
          product_step(more[i & 1][o], f.kt[o][i], u[i], r);
#pragma unroll
      for (int o = 0; o < OWN; ++o)
        if (i > 0) S[o] += more[(i - 1) & 1][o][0] + more[(i - 1) & 1][o][1];
      fetch_kt(ahead, later, i);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) S[o] += more[1][o][0] + more[1][o][1];
  };
  WalkOperands<NT> ring[4];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) fetch_w(ring[i], unit_of(begin + i), j);
#pragma unroll
    for (int j = 0; j < 4; ++j) fetch_kt(ring[i], unit_of(begin + i), j);
  }
  for (int chunk = begin; chunk < end; chunk += 4) {
    turn(ring[0], ring[3], chunk);
    if (chunk + 1 < end) turn(ring[1], ring[0], chunk + 1);
    if (chunk + 2 < end) turn(ring[2], ring[1], chunk + 2);
    if (chunk + 3 < end) turn(ring[3], ring[2], chunk + 3);
  }
#pragma unroll
  for (int o = 0; o < OWN; ++o)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * (w + 4 * o) + 4 * g + r;
      if (n < a.N && p < a.P) st[(int64_t)n * a.P + p] = S[o][r];
    }
}

// ---------------------------------------------------------------- o
// A workgroup takes one chunk and `heads_each` heads that read the same q and k (their products
// are made once); a wavefront takes every fourth tile of 16 columns.
template <int NT, bool DELTA, bool ROW, int FORM, int RT>
__device__ __forceinline__ void output_chunk(const ChunkedArgs& a, const ChunkRange& c, int heads_each,
                                             int wide) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  extern __shared__ __align__(16) float lds[];
  float* Qs = lds;
  float* Ks = Qs + kTok * LD;
  float* Gs = Ks + kTok * LD;                             // ROW only
  float* tiles = ROW ? Gs + kTok * LD : Ks;               // (else in the keys' place, once they are read)
  float* blocks = tiles + kTiles * kTile;                 // ROW: [4][NP]
  float* decays = blocks;                                 // else [heads_each] of HeadDecays
  const int chunk = blockIdx.y, h0 = blockIdx.x * heads_each;
  const int hk = h0 / (a.heads / a.kv_heads), PT = (a.P + 15) / 16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, l = lane % 16, g = lane / 16;
  const Parts parts = parts_of(a.num_chunks, a.heads, a.N, a.P, DELTA);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  float dec[2] = {1.f, 1.f}, vs[2] = {0.f, 0.f};          // of heads w and w + 4, a token a lane
  if (!ROW) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (w + 4 * u < heads_each && lane < c.nt)
        token_scalars(a, c.first + lane, h0 + w + 4 * u, dec[u], vs[u]);
  }
  stage_rows<NP, FORM>(a, Qs, a.q_col + hk * a.N, c.first, c.nt, c.pos0, false, wide);
  stage_rows<NP, FORM>(a, Ks, a.k_col + hk * a.N, c.first, c.nt, c.pos0, true, wide);
  if (ROW) stage_decays<NP>(a, Gs, h0, c.first, c.nt);
  __syncthreads();
  f32x4 gram[3];
  if (ROW) {
    if (w < RT) diagonal_tiles<NP, false>(tiles, Qs, Ks, Gs, w, lane);
    __syncthreads();
    split_decays<NP>(Qs, Ks, Gs, blocks);
    __syncthreads();
    for (int t = w; t < kTiles; t += 4) {
      const int i = tri_row(t), j = t - tri(i, 0);
      if (i >= RT) break;
      if (i == j) continue;
      const f32x4 acc = split_tile<NT>(Qs, Gs, blocks, i, j, l, g);
#pragma unroll
      for (int r = 0; r < 4; ++r) tiles[t * kTile + (4 * g + r) * kTileLd + l] = acc[r];
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int t = w + 4 * u, i = tri_row(t), j = t - tri(i, 0);
      if (t < kTiles && i < RT) gram[u] = gram_tile<NT>(Qs + 16 * i * LD, Ks + 16 * j * LD, l, g);
    }
    __syncthreads();                       // the keys have been read
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (w + 4 * u < heads_each)
        spread_decays(HeadDecays{decays + (w + 4 * u) * HeadDecays::kFloats}, dec[u], vs[u], lane);
  }
  for (int h = h0; h < h0 + heads_each; ++h) {
    const int64_t unit = (int64_t)chunk * a.heads + h;
    const HeadDecays d{decays + (h - h0) * HeadDecays::kFloats};
    if (!ROW) {
      __syncthreads();                     // the decays are there; the head before has been read
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const int t = w + 4 * u, i = tri_row(t), j = t - tri(i, 0);
        if (t < kTiles && i < RT) {
          const f32x4 m = tile_decays(d, i, j, l, g);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            tiles[t * kTile + (4 * g + r) * kTileLd + l] = i > j || 4 * g + r >= l ? gram[u][r] * m[r] : 0.f;
        }
      }
      __syncthreads();
    }
    const float skip = a.d_skip ? a.d_skip[h] : 0.f;
    for (int ct = w; ct < PT; ct += 4) {
      // (unknown to the compiler in every turn, or it keeps the comparisons with them, and all of
      // q, in registers from turn to turn and runs out of both kinds)
      int nt = c.nt;
      asm volatile("" : "+v"(nt)::"memory");
      const int p = 16 * ct + l;
      const float* start = a.scratch + parts.starts + (unit * PT + ct) * NT * 256 + lane * 4;
      f32x4 s0[NT], v[RT];                 // v as it stands, or u
#pragma unroll
      for (int j = 0; j < NT; ++j) s0[j] = read4(start + j * 256);
      if (DELTA) {
#pragma unroll
        for (int j = 0; j < RT; ++j)
          v[j] = read4(a.scratch + parts.u + ((unit * PT + ct) * 4 + j) * 256 + lane * 4);
      } else {
        const float* col = a.x + (int64_t)c.first * a.ld + a.v_col + h * a.P + p;
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 16 * j + 4 * g + r;
            v[j][r] = t < nt && p < a.P ? col[(int64_t)t * a.ld] : 0.f;
          }
      }
      f32x4 acc[RT], part[2][RT][2], q[2][RT];
      auto fetch = [&](int j) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          q[j & 1][i] = read4(Qs + (16 * i + l) * LD + 16 * j + 4 * g);
          if (ROW)
            for (int m = 0; m < i; ++m) q[j & 1][i] *= read4(blocks + m * NP + 16 * j + 4 * g);
        }
      };
      fetch(0);
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] = zero;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (j + 1 < NT) fetch(j + 1);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int i = 0; i < RT; ++i)
            product_step(part[j & 1][i], q[j & 1][i], s0[j], r);
        // (the sixteen before are added meanwhile; put off to the end by the compiler otherwise, which
        // then has no registers left)
        if (j > 0) {
#pragma unroll
          for (int i = 0; i < RT; ++i) {
            acc[i] += part[(j - 1) & 1][i][0] + part[(j - 1) & 1][i][1];
            asm volatile("" : "+v"(acc[i]));
          }
        }
        __builtin_amdgcn_sched_group_barrier(8, 3, 0);
#pragma unroll
        for (int m = 3; m < 4 * RT; ++m) {
          __builtin_amdgcn_sched_group_barrier(8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(2, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] += part[(NT - 1) & 1][i][0] + part[(NT - 1) & 1][i][1];
      if (FORM == kSilu) {
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[j][r] = silu(v[j][r]);
      }
      float* out = a.out + (int64_t)c.first * a.heads * a.P + h * a.P + p;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        if (!ROW) acc[i] *= read4(d.d0() + 16 * i + 4 * g);
        f32x4 pair = zero;
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          const f32x4 t = read4(tiles + tri(i, j) * kTile + l * kTileLd + 4 * g);
          const f32x4 p = i == j ? causal_product(t, v[j], g) : product2(t, v[j]);
          pair = j & 1 ? pair + p : p;
          if (j & 1 || j == i) acc[i] += pair;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * i + 4 * g + r;
          if (t < nt && p < a.P)
            out[(int64_t)t * a.heads * a.P] = DELTA ? acc[i][r] : fmaf(skip, v[i][r], acc[i][r]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <int NT, bool DELTA, bool ROW, int FORM>
__global__ __launch_bounds__(kThreads, 2) void chunk_output_kernel(ChunkedArgs a, int heads_each, int wide) {
  const ChunkRange c = chunk_range(a, blockIdx.y);
  if (c.tiles == 1) output_chunk<NT, DELTA, ROW, FORM, 1>(a, c, heads_each, wide);
  else output_chunk<NT, DELTA, ROW, FORM, 4>(a, c, heads_each, wide);
}

template <typename F>
bool raise_lds(F* fn, size_t bytes) {
  return bytes <= 64 * 1024 ||
         hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

template <int NT, bool DELTA, bool ROW, int FORM>
int launch_output(const ChunkedArgs& a, int heads_each, int wide, hipStream_t stream) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  const int keys = ROW ? 2 * kTok * LD + kTiles * kTile + 4 * NP
                       : std::max(kTok * LD, kTiles * kTile + heads_each * HeadDecays::kFloats);
  const size_t lds = sizeof(float) * (kTok * LD + keys);
  auto* fn = chunk_output_kernel<NT, DELTA, ROW, FORM>;
  if (!raise_lds(fn, lds)) return -1;
  hipLaunchKernelGGL(fn, dim3(a.heads / heads_each, a.num_chunks), dim3(kThreads), lds, stream, a,
                     heads_each, wide);
  return 0;
}

// Whether linear forms go in two launches, which walk 64 tokens in 2.3 us (up to 64 rows of S: 1.4)
// whatever else the chip does, or in three, whose work is spread over it: us in two and three launches,
// 256 workgroups in the walk (64 heads of 128 x 64) 170 tokens 26 / 35, 1,000 63 / 80, 2,048 98 / 123,
// 8,192 360 / 464; 128 (16 heads of 128 x 128) 300 tokens 30 / 44, 1,000 55 / 55, 2,048 93 / 84;
// 64 (16 heads of 64 x 64) 300 tokens 20 / 26, 1,000 39 / 29.  The longest portion of a step decides for
// all of its requests, whose results do not hang on it: both give the same bits.  (More rows than 128 do not fit the walk's
// registers; an output's place in a chunk is counted in 32 bits.)
bool in_two_launches(const ChunkedArgs& a) {
  const int64_t chunks = (a.max_len + kTok - 1) / kTok;
  return a.N <= 128 && (int64_t)a.heads * a.P <= 1 << 22 &&
         (int64_t)a.heads * ((a.P + 15) / 16) >= 8 * std::min<int64_t>(chunks, 32);
}

template <int NT, int FORM>
int launch_scan(const ChunkedArgs& a, int each, int wide, hipStream_t stream) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  const size_t lds = sizeof(float) * (2 * kTok * LD + each * HeadDecays::kFloats);
  auto* prepare = chunk_prepare_kernel<NT, FORM>;
  if (!raise_lds(prepare, lds)) return -1;
  hipLaunchKernelGGL(prepare, dim3(a.heads / each, a.num_chunks), dim3(kThreads), lds, stream, a, each, wide);
  hipLaunchKernelGGL((chunk_scan_kernel<NT, FORM>), dim3(a.heads, (a.P + 15) / 16, a.num_entries),
                     dim3(kScanThreads), 0, stream, a);
  return 0;
}

template <int NT, int FORM>
int launch_linear(const ChunkedArgs& a, int wide, hipStream_t stream) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  // heads that share q and k share a workgroup as long as there are two workgroups a unit
  int each = a.heads / a.kv_heads;
  while (each % 2 == 0 && (each > 8 || (int64_t)(a.heads / each) * a.num_chunks < 512)) each /= 2;
  if (each > 8) each = 1;
  if constexpr (NT <= 8)
    if (in_two_launches(a)) return launch_scan<NT, FORM>(a, each, wide, stream);
  const size_t lds = sizeof(float) * (kTok * LD + kTok * 68 + each * kTok);
  auto* local = chunk_local_kernel<NT, FORM>;
  if (!raise_lds(local, lds)) return -1;
  const int PT = (a.P + 15) / 16;
  hipLaunchKernelGGL(local, dim3(a.heads / each, a.num_chunks), dim3(kThreads), lds, stream, a, each, wide);
  hipLaunchKernelGGL(chunk_carry_kernel<NT>, dim3(a.heads, a.num_entries, (PT * NT * 64 + kThreads - 1) / kThreads),
                     dim3(kThreads), 0, stream, a);
  return launch_output<NT, false, false, FORM>(a, each, wide, stream);
}

template <int NT>
int launch_form(const ChunkedArgs& a, int wide, hipStream_t stream) {
  return a.turn   ? launch_linear<NT, kTurned>(a, wide, stream)
         : a.silu ? launch_linear<NT, kSilu>(a, wide, stream)
                  : launch_linear<NT, kPlain>(a, wide, stream);
}

template <int NT, bool ROW>
int launch_delta(const ChunkedArgs& a, int wide, hipStream_t stream) {
  constexpr int NP = 16 * NT, LD = NP + 4;
  const size_t lds = sizeof(float) * ((ROW ? 2 : 1) * kTok * LD + kTiles * kTile + kTok + (ROW ? 4 * NP : HeadDecays::kFloats));
  auto* solve = chunk_solve_kernel<NT, ROW>;
  if (!raise_lds(solve, lds)) return -1;
  hipLaunchKernelGGL(solve, dim3(a.heads, a.num_chunks), dim3(kThreads), lds, stream, a, wide);
  hipLaunchKernelGGL(chunk_walk_kernel<NT>, dim3(a.heads, a.num_entries, (a.P + 15) / 16), dim3(kThreads),
                     0, stream, a);
  return launch_output<NT, true, ROW, kPlain>(a, 1, wide, stream);
}

}  // namespace

int64_t chunked_scratch_floats(int num_chunks, int heads, int kv_heads, int N, int P, int delta) {
  if (N < 1 || P < 1 || N > (delta ? 128 : 256)) return -1;
  const int64_t end = parts_of(num_chunks, heads, N, P, delta).end;
  return delta ? end : std::max(end, scan_parts_of(num_chunks, heads, kv_heads, N).end);
}

extern "C" int64_t ts_chunked_scratch(int num_chunks, int heads, int kv_heads, int N, int P, int delta) {
  return chunked_scratch_floats(num_chunks, heads, kv_heads, N, P, delta);
}

extern "C" int ts_chunk_tokens() { return kChunkTokens; }

int launch_chunked(ChunkedArgs a, hipStream_t stream) {
  if (chunked_scratch_floats(a.num_chunks, a.heads, a.kv_heads, a.N, a.P, a.delta) < 0)
    TS_FAIL("chunked recurrence: %d rows of S are not built", a.N);
  if (a.num_chunks > 65535 || a.num_entries > 65535 || a.P > 1 << 19)
    TS_FAIL("chunked recurrence: %d chunks, %d entries, %d columns", a.num_chunks, a.num_entries, a.P);
  if ((a.turn || a.silu) && (a.delta || (a.turn && a.silu)))
    TS_FAIL("chunked recurrence: SiLU or a rotation of the operands, and without the delta rule");
  const int wide = a.N % 4 == 0 && a.ld % 4 == 0 && a.q_col % 4 == 0 && a.k_col % 4 == 0 &&
                   ((uintptr_t)a.x & 15) == 0;
  int rc;
  if (a.delta && a.per_row)
    rc = a.N <= 32 ? launch_delta<2, true>(a, wide, stream)
       : a.N <= 64 ? launch_delta<4, true>(a, wide, stream) : launch_delta<8, true>(a, wide, stream);
  else if (a.delta)
    rc = a.N <= 32 ? launch_delta<2, false>(a, wide, stream)
       : a.N <= 64 ? launch_delta<4, false>(a, wide, stream) : launch_delta<8, false>(a, wide, stream);
  else
    rc = a.N <= 32 ? launch_form<2>(a, wide, stream) : a.N <= 64 ? launch_form<4>(a, wide, stream)
       : a.N <= 128 ? launch_form<8>(a, wide, stream) : launch_form<16>(a, wide, stream);
  if (rc != 0) TS_FAIL("chunked recurrence: %d rows of S need more LDS than the device gives", a.N);
  TS_CHECK_LAUNCH("chunked recurrence");
  return 0;
}
