// The kernel of 32 rows a wavefront for scores with extras (attention.h).
#include "attention_prefill_tall_kernel.h"

template <int HD>
static int launch(const AttentionMfmaArgs& args, hipStream_t stream) {
  switch (args.sets) {
    case 1: return launch_prefill_tall<HD, 4, 1, 64, true>(args, stream);
    case 2: return launch_prefill_tall<HD, 4, 2, 64, true>(args, stream);
    case 4: return launch_prefill_tall<HD, 2, 4, 32, true>(args, stream);
  }
  TS_FAIL("attention_prefill: no form of %d sets", args.sets);
}

int launch_attention_prefill_tall_scores(const AttentionMfmaArgs& args, hipStream_t stream) {
  return args.base.hd == 64 ? launch<64>(args, stream) : launch<128>(args, stream);
}
