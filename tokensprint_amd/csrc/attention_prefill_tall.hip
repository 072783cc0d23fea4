#include "attention_prefill_tall_kernel.h"

template <int HD>
static int launch(const AttentionMfmaArgs& args, hipStream_t stream) {
  switch (args.sets) {
    case 1: return launch_prefill_tall<HD, 4, 1, 64, false>(args, stream);
    case 2: return launch_prefill_tall<HD, 4, 2, 64, false>(args, stream);
    case 4: return launch_prefill_tall<HD, 2, 4, 32, false>(args, stream);
  }
  TS_FAIL("attention_prefill: no form of %d sets", args.sets);
}

int launch_attention_prefill_tall_scores(const AttentionMfmaArgs& args, hipStream_t stream);

// Items of four tiles for four sets, of eight for one and two.
int launch_attention_prefill_tall(const AttentionMfmaArgs& args, hipStream_t stream) {
  if (has_score_extras(args.base)) return launch_attention_prefill_tall_scores(args, stream);
  return args.base.hd == 64 ? launch<64>(args, stream) : launch<128>(args, stream);
}
