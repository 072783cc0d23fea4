// The two halves of a prompt's layer as one call each: their kernels one behind the other on the
// stream, with no return to the caller in between.  An eager step of few rows waits for the host, whose
// share of a call (arguments, checks, outputs) is twice the launch itself: 0.6B, a prompt of 300 tokens,
// 1.87 -> 1.74 ms a step.
#include "attention_mfma.h"
#include "qk_prepare.h"

extern "C" int ts_gemm_tiled_heads_bf16(const void* rows, const float* sumsq, int parts, float eps, const void* w,
                                        const QkPrepareArgs* heads, int M, int K, int tile, hipStream_t stream);
extern "C" int ts_gemm_tiled_tail_bf16(const void* a, const void* w, float* resid, const float* norm_w,
                                       void* prepared, float* sumsq, int M, int N, int K, int tile,
                                       hipStream_t stream);
extern "C" int ts_gemm_tiled_scaled_bf16(const void* rows, const float* sumsq, int parts, float eps, const void* w,
                                         void* c, int c_type, int M, int N, int K, int pair, int tile,
                                         hipStream_t stream);
extern "C" int ts_attention_prefill(const AttentionMfmaArgs* args, hipStream_t stream);
extern "C" int ts_attention_mfma(const AttentionMfmaArgs* args, hipStream_t stream);

// rows[M, K] and sumsq[parts, M]: what the product before has prepared; resid[M, N], norm_w[N],
// prepared[M, N] and sumsq_out: the stream, the next norm, and what is prepared for it.
struct PromptStream {
  const void* rows;
  const float* sumsq;
  float* resid;
  const float* norm_w;
  void* prepared;
  float* sumsq_out;
  int parts, M, K, N;
  float eps;
};

struct PromptAttentionArgs {
  PromptStream s;
  const void *w_qkv, *w_o;
  QkPrepareArgs heads;
  AttentionMfmaArgs attention;      // its queries are the heads' q_out
  int prefill;                      // the kernel for long portions (ts_attention_prefill)
};

// ts_gemm_tiled_heads_bf16, attention, ts_gemm_tiled_tail_bf16.
extern "C" int ts_prompt_attention(const PromptAttentionArgs* p, hipStream_t stream) {
  const PromptStream& s = p->s;
  const AttentionArgs& a = p->attention.base;
  if (a.q != p->heads.q_out || a.num_tokens != s.M || a.nq != p->heads.nq || a.hd != p->heads.hd)
    TS_FAIL("prompt_attention: attention over other queries than the projection's");
  if (ts_gemm_tiled_heads_bf16(s.rows, s.sumsq, s.parts, s.eps, p->w_qkv, &p->heads, s.M, s.K, 0, stream)) return -1;
  if (p->prefill ? ts_attention_prefill(&p->attention, stream) : ts_attention_mfma(&p->attention, stream)) return -1;
  return ts_gemm_tiled_tail_bf16(a.out, p->w_o, s.resid, s.norm_w, s.prepared, s.sumsq_out, s.M, s.N,
                                 a.nq * a.hd, 0, stream);
}

// ts_gemm_tiled_scaled_bf16 of w_gate_up[2 I, K] into act[M, I], ts_gemm_tiled_tail_bf16 of w_down[N, I].
extern "C" int ts_prompt_feed_forward(const PromptStream* p, const void* w_gate_up, const void* w_down,
                                      void* act, int I, hipStream_t stream) {
  const PromptStream& s = *p;
  if (ts_gemm_tiled_scaled_bf16(s.rows, s.sumsq, s.parts, s.eps, w_gate_up, act, TS_BF16, s.M, I, s.K, 1, 0, stream))
    return -1;
  return ts_gemm_tiled_tail_bf16(act, w_down, s.resid, s.norm_w, s.prepared, s.sumsq_out, s.M, s.N, I, 0, stream);
}
