"""Float32 attention at the edges of its kernel: blocks of 16 keys over eight wavefronts, and more tiles
than the grid's second dimension takes at once."""

import pytest
import torch

from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def attended(ops, device, spans, nq, nkv, hd, window, page=16):
    """(result, float64 queries by entry, keys, values [nkv, positions, hd] by entry)"""
    batch, cache, table, _ = paged_scenario(device, torch.float32, nkv=nkv, hd=hd, page_size=page, spans=spans)
    q = rand((batch.num_tokens, nq, hd), 1).to(device)
    out = ops.paged_attention(q, batch, table, cache, num_heads=nq, num_kv_heads=nkv, head_dim=hd,
                              scale=hd ** -0.5, window=window)
    keys, values = [], []
    for entry, (start, count) in enumerate(spans):
        pages = table[entry].long().clamp(min=0)
        keys.append(cache.k_pages[pages].double().permute(1, 0, 2, 3).reshape(nkv, -1, hd)[:, :start + count])
        values.append(cache.v_pages[pages].double().permute(1, 0, 3, 2).reshape(nkv, -1, hd)[:, :start + count])
    return out, q.double(), keys, values


# first and last key of a block of a wavefront, of the eighth wavefront, of its second and third turn
@pytest.mark.parametrize("window", [None, 17])
@pytest.mark.parametrize("nq, nkv, hd", [(4, 2, 128), (3, 3, 16), (6, 1, 96)])
def test_edges_of_blocks_and_turns(gpu_device, nq, nkv, hd, window):
    spans = [(0, 1), (15, 1), (16, 1), (127, 2), (128, 1), (255, 3), (0, 40), (383, 5)]
    out, q, keys, values = attended(load_hip_ops(gpu_device), gpu_device, spans, nq, nkv, hd, window)
    row = 0
    for (start, count), k, v in zip(spans, keys, values):
        k, v = (x.repeat_interleave(nq // nkv, 0) for x in (k, v))
        scores = torch.matmul(q[row:row + count].permute(1, 0, 2), k.transpose(1, 2).contiguous()) * hd ** -0.5
        behind = (start + torch.arange(count, device=gpu_device))[:, None] - torch.arange(
            start + count, device=gpu_device)[None]
        scores.masked_fill_((behind < 0) | (behind >= (window or 1 << 30)), float("-inf"))
        want = torch.matmul(scores.softmax(-1), v).permute(1, 0, 2)
        # scores: hd products and two roundings of up to |s| ~ 5; values: a sum of weights that are one together
        assert (out[row:row + count].double() - want).abs().max() < 2 ** -23 * (5 * 5 + 8) * 4
        row += count


def test_more_tiles_than_one_grid_dimension(gpu_device):
    """16 query heads a key/value head: a tile a token, 33,000 of them."""
    T, hd, window = 33_000, 16, 16
    out, q, (k,), (v,) = attended(load_hip_ops(gpu_device), gpu_device, [(0, T)], 16, 1, hd, window, page=64)
    for first in (0, 32_768 - 20, T - 300):
        tokens = torch.arange(first, first + 300 if first else 300, device=gpu_device).clamp(max=T - 1)
        seen = tokens[:, None] - torch.arange(window, device=gpu_device)[None]         # [300, 16]
        at = seen.clamp(min=0)
        scores = (q[tokens][:, :, None] * k[0][at][:, None]).sum(-1) * hd ** -0.5      # [300, heads, 16]
        scores.masked_fill_(seen[:, None] < 0, float("-inf"))
        want = (scores.softmax(-1)[..., None] * v[0][at][:, None]).sum(2)
        assert (out[tokens].double() - want).abs().max() < 2 ** -23 * (5 * 5 + 8) * 4
