"""bench.py's split of a step: with one kind of call made empty no kernel of that kind runs, whichever
calls the step is made of."""

import pytest

import bench
from helpers import qwen3_config
from tokensprint_amd.engine.assemble import random_model
from tokensprint_amd.engine.runner import ModelRunner

pytestmark = pytest.mark.gpu
#: what the names of library functions of a kind hold; the preparation of q, k and v is attention's
KINDS = {"attention": ("attention", "qk_prepare", "tiled_heads"), "products": ("gemm", "prompt")}


# a sub-layer as one call, a long portion too; calls one by one
@pytest.mark.parametrize("tokens", [300, 600, 40])
def test_nothing_of_a_kind_runs_without_it(gpu_device, monkeypatch, tokens):
    cfg = qwen3_config(hidden=1024, layers=2, heads=8, kv_heads=4, head_dim=128, inter=1536, vocab=512,
                       eps=1e-6, theta=1e4, tied=True, max_pos=1024)
    _, model = random_model(cfg, 0)
    ops, called = model.ctx.ops, []
    call = ops._call
    monkeypatch.setitem(vars(ops), "_call", lambda fn, *args: (called.append(fn.__name__), call(fn, *args))[1])

    def step():
        runner = ModelRunner(model, page_size=16, num_pages=tokens // 16 + 2, num_slots=1)
        batch = runner.build(bench.prefill_entries(tokens)(runner))
        called.clear()
        runner.run(batch)
        return list(called)

    def of(kind, names):
        return [n for n in names if any(part in n for part in KINDS[kind])]

    whole = step()
    assert ("ts_prompt_attention" in whole) == (tokens > 64)
    for kind in KINDS:
        assert of(kind, whole)
        with bench.Without(ops, kind):
            assert of(kind, step()) == []
        assert not set(bench.ATTENTION + bench.PRODUCTS) & set(vars(ops))
        assert step() == whole
