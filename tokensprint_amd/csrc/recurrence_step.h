// Recurrences of a step in which every entry brings one token (recurrence_step.hip): what the
// entry points that walk entries of any length hand over.
#pragma once
#include "common.h"

// The operands of token e, which is entry e's only one.
struct RecurrenceStepArgs {
  const float* x;        // [T, ld]: q (kv_heads*N) at q_col, k at k_col, v (heads*P) at v_col
  const float* decay;    // [heads]: the fixed decays, or null
  const float* gates;    // [T, ldg]: beta (heads) | g (heads, or heads*N), or null
  float* state;          // [slots, heads, N, P]
  float* out;            // [T, heads*P]
  const int *positions, *slot_ids;
  int ld, q_col, k_col, v_col, ldg, heads, kv_heads, N, P, silu;
  const float2* turn;    // [max_pos, turn_dims / 2], or null
  int turn_dims;
  float k_scale;
  // from the projections to the gated rows in one kernel (delta rule; `gated` set): q and k are
  // made unit vectors, beta and g made on the way, and the head's output is normed and gated
  const float *beta, *z, *a_log, *dt_bias;   // rows of ldb and ldz
  const float *gate, *norm_w;                // gate rows of ldgate; norm_w [P]
  void* gated;                               // [T, heads*P]
  int ldb, ldz, ldgate, act;                 // act 0: sigmoid, 1: SiLU
  float eps;
};

// Whether the kernel takes these operands (sizes, places); without `gated`.
bool recurrence_step_fits(const RecurrenceStepArgs& a);
void launch_recurrence_step(const RecurrenceStepArgs& a, int num_entries, bool delta, bool per_row,
                            hipStream_t stream);

struct ScanStepArgs {
  const float* xbc;       // [T, channels]: x (heads*P) | B (groups*N) | C (groups*N)
  const float* dt;        // [T, ldt]: a step size per head
  const float *dt_bias, *a_log, *d_skip;     // [heads]
  float* state;           // [slots, heads, N, P]
  float* y;               // [T, heads*P]
  const int *positions, *slot_ids;
  int ldt, heads, P, N, groups;
};

bool scan_step_fits(const ScanStepArgs& a);
void launch_scan_step(const ScanStepArgs& a, int num_entries, hipStream_t stream);
