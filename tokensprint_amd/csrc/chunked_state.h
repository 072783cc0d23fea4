// The recurrences of matrix_state.hip and ssm.hip in chunks of 64 tokens (chunked_state.hip).
#pragma once
#include "common.h"

struct BatchView {
  const int* positions;       // [T]
  const int* entry_of_token;  // [T]
  const int* q_start;         // [B + 1]
  const int* slot_ids;        // [B]
};

constexpr int kChunkTokens = 64;

// S <- g S;  u = vs v, or (delta) beta (vs v - S^T k);  S <- S + k u^T;  o = S^T q (+ skip v),
// per head and entry, float32.  Which of the forms is said by the pointers that are set.
struct ChunkedArgs {
  const float* x;             // [T, ld]: q at q_col, k at k_col (kv_heads x N), v (heads x P) at v_col
  float* state;               // [slots, heads, N, P]
  float* out;                 // [T, heads * P]
  BatchView b;
  int ld, q_col, k_col, v_col, heads, kv_heads, N, P, silu;
  // g: a fixed decay a head; or gates [T, ldg], beta (heads) | g (heads, or per_row heads x N);
  // or from a step size d = softplus(dt + dt_bias): g = exp(-exp(a_log) d), vs = d
  const float* decay;
  const float* gates;
  const float* dt;            // [T, ldg], heads columns from its first
  const float *dt_bias, *a_log, *d_skip;
  int ldg, delta, per_row;
  const float2* turn;         // [positions, turn_dims / 2], or null
  int turn_dims;
  float k_scale;
  // every entry in runs of 64 tokens, the last of them shorter
  const int* chunks;          // [num_chunks, 3]: first token, one past the last, entry
  const int* entry_chunks;    // [B + 1]
  int num_chunks, num_entries;
  int max_len;                // the most tokens an entry brings
  float* scratch;             // chunked_scratch_floats of them, 16-byte aligned
};

// Floats of scratch that launch_chunked wants; -1: these sizes are not built in chunks.
int64_t chunked_scratch_floats(int num_chunks, int heads, int kv_heads, int N, int P, int delta);
int launch_chunked(ChunkedArgs a, hipStream_t stream);
