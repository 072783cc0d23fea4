"""What a block with a token shift tells the block in front: in steps of single tokens the norm and
the shift behind its last add, in others nothing, so that a portion's layers do no work for it.
On the CPU, with the plain torch kernel references and the fused call beside them."""

import torch

import drives
from helpers import ZONO_A, random_prompt
from kernel_refs import TorchOps
from tokensprint_amd.engine import ModelRunner
from tokensprint_amd.engine.assemble import load_model
from tokensprint_amd.kernels import stream
from tokensprint_amd.weights import write_random_model


class FusedOps(TorchOps):
    def __init__(self):
        super().__init__()
        self.steps = []

    def postnorm_add_shift(self, resid, delta, post_w, post_eps, norm_w, norm_eps, shift_w, batch,
                           state, out_dtype):
        self.steps.append((batch.max_q_len, batch.num_tokens, batch.num_entries))
        self.postnorm_add(resid, delta, post_w, post_eps)
        return self.norm_token_shift(resid, norm_w, norm_eps, shift_w, batch, state, out_dtype)


def test_only_steps_of_single_tokens_ask_for_the_shift(tmp_path, monkeypatch):
    write_random_model(tmp_path, ZONO_A, 1, torch.float32, std=0.2)
    requests = {f"r{i}": random_prompt(n, ZONO_A["vocab"], 40 + i) for i, n in enumerate((9, 1, 40))}
    made, init = [], stream.ShiftAhead.__init__
    monkeypatch.setattr(stream.ShiftAhead, "__init__",
                        lambda self, *a, **k: made.append(self) or init(self, *a, **k))

    def logits(ops):
        _, model = load_model(tmp_path, "float32", "cpu", ops=ops)
        runner = ModelRunner(model, page_size=8, num_pages=12, num_slots=4)
        return drives.drive_prefill_then_decode(runner, requests), model

    want, _ = logits(TorchOps())
    assert not made
    ops = FusedOps()
    got, model = logits(ops)
    assert ops.steps and all(q == 1 and tokens == entries for q, tokens, entries in ops.steps)
    assert len(made) == len(ops.steps)
    for rid in requests:
        assert torch.equal(got.stacked(rid)[0], want.stacked(rid)[0])
    # the entry hints are made with the blocks
    assert all(block.entry_hint() is block.entry_hint() for block in model.blocks)
