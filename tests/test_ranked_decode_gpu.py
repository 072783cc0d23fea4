"""Decode attention whose items are ranked by their contexts (more items than compute units, one split):
which workgroup takes an entry changes no bit of what it makes, so halves of the entries, which are not
ranked, come out the same."""

import pytest
import torch

from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu


def lengths(kind, count):
    if kind == "equal":
        return [77] * count
    if kind == "falling":
        return [40 * (count - i) for i in range(count)]
    return [1 + (i * 7919) % 1500 // (1 + i % 3) for i in range(count)]       # ragged, some alike, some 1


@pytest.mark.parametrize("kind", ["equal", "falling", "ragged"])
@pytest.mark.parametrize("count, nkv, group, hd, window", [
    (64, 8, 2, 128, None), (64, 5, 1, 64, 100), (33, 8, 4, 128, None), (40, 7, 2, 32, 64)])
def test_ranked_items_are_the_same_items(gpu_device, count, nkv, group, hd, window, kind):
    ops, nq = load_hip_ops(gpu_device), nkv * group
    assert count * nkv > 256 and (count + 1) // 2 * nkv <= 256
    spans = [(n - 1, 1) for n in lengths(kind, count)]
    gen = torch.Generator().manual_seed(3)
    rows = torch.randn(count, (nq + 2 * nkv) * hd, generator=gen).to(gpu_device, torch.bfloat16)
    angles = 40 * torch.randn(3000, hd // 2, generator=gen)
    weight = (1 + 0.1 * torch.randn(hd, generator=gen)).to(gpu_device)
    kw = dict(num_heads=nq, num_kv_heads=nkv, kv_in_row=nkv, head_dim=hd, q_weight=weight, k_weight=weight,
              eps=1e-6, cos_sin=(angles.cos().to(gpu_device), angles.sin().to(gpu_device)),
              scale=hd ** -0.5, window=window)

    def step(parts):
        batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=nkv, hd=hd, page_size=16,
                                                spans=spans)
        outs = []
        for part in parts:
            sub = Part(batch, part) if len(part) < count else batch
            outs.append(ops.attend(rows[part].contiguous(), sub, table[part].contiguous(), cache, True, **kw))
        return torch.cat(outs), cache.k_pages, cache.v_pages

    every, half = list(range(count)), (count + 1) // 2
    # (one split in halves as in the whole: key splits would add up in another order)
    ops._decode_splits = lambda items, span: 1
    try:
        whole, k_whole, v_whole = step([every])
        parts, k_parts, v_parts = step([every[:half], every[half:]])
    finally:
        del ops._decode_splits
    assert torch.equal(whole, parts)
    assert torch.equal(k_whole, k_parts) and torch.equal(v_whole, v_parts)


class Part:
    """Some entries of a batch of single tokens."""

    def __init__(self, batch, entries):
        def of(t):
            return t[entries].contiguous()
        self.positions, self.ctx_len = of(batch.positions), of(batch.ctx_len)
        count = len(entries)
        self.entry_of_token = torch.arange(count, dtype=torch.int32, device=batch.positions.device)
        self.q_start = torch.arange(count + 1, dtype=torch.int32, device=batch.positions.device)
        self.num_tokens = self.num_entries = count
        self.max_q_len, self.max_ctx_len = 1, batch.max_ctx_len
        self.q_lens, self.plans = [1] * count, {}
