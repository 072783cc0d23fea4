"""The halves of a prompt's layer as one call each, against their kernels called one by one: the same
kernels, so the same bits, in the stream, the rows prepared for the next norm and the pages."""

import dataclasses

import pytest
import torch

from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.kernels.stream import NormHint, PreparedRows

pytestmark = pytest.mark.gpu
EPS, NQ, NKV, HD, D, INNER = 1e-6, 8, 4, 128, 1024, 1536


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def prepared(device, T, weight, silu_mul=False):
    hint = NormHint(torch.ones(D, device=device), EPS, weight, silu_mul)
    sumsq = (rand((D // 32, T), 3).square() * 20 + 1).to(device)
    return PreparedRows(rand((T, D), 2).to(device, torch.bfloat16), sumsq, D // 32, hint, tiled=True)


def same(got, want, stream, other):
    assert torch.equal(got.rows, want.rows) and torch.equal(got.sumsq, want.sumsq)
    assert got.slices == want.slices and got.tiled and got.hint is want.hint
    assert torch.equal(stream, other)


@pytest.mark.parametrize("window, softcap", [(None, None), (40, None), (None, 30.0)])
@pytest.mark.parametrize("spans", [
    [(0, 72)], [(0, 257)], [(3, 129), (0, 1), (100, 60)], [(700, 72), (900, 72)], [(0, 700), (5, 300)]])
def test_attention_in_one_call(gpu_device, spans, window, softcap):
    ops = load_hip_ops(gpu_device)
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=NKV, hd=HD, page_size=16,
                                            spans=spans)
    other = dataclasses.replace(cache, k_pages=cache.k_pages.clone(), v_pages=cache.v_pages.clone())
    w_qkv, w_o, w_next = ((0.05 * rand(shape, i)).to(gpu_device, torch.bfloat16) for i, shape in enumerate(
        [((NQ + 2 * NKV) * HD, D), (D, NQ * HD), (2 * INNER, D)]))
    delta = prepared(gpu_device, batch.num_tokens, w_qkv)
    stream = rand((batch.num_tokens, D), 4).to(gpu_device)
    expected = stream.clone()
    hint = NormHint(torch.ones(D, device=gpu_device), EPS, w_next, True)
    angles = 40 * rand((1200, HD // 2), 5)
    norms = [(1 + 0.1 * rand((HD,), i)).to(gpu_device) for i in (6, 7)]
    heads = dict(num_heads=NQ, num_kv_heads=NKV, head_dim=HD)
    kinds = dict(q_weight=norms[0], k_weight=norms[1], head_eps=EPS,
                 cos_sin=(angles.cos().to(gpu_device), angles.sin().to(gpu_device)))
    scores = dict(scale=HD ** -0.5, window=window, softcap=softcap)
    norm_w = delta.hint.norm_weight
    got = ops.attend_into_stream(stream, delta, norm_w, EPS, w_qkv, batch, table, cache, w_o, hint,
                                 **heads, **kinds, **scores)
    q = ops.norm_heads(expected, delta, norm_w, EPS, w_qkv, batch, table, other, **heads, **kinds, tile=2)
    if got is None:                        # the projection on its own is the faster way there
        assert torch.equal(stream, expected)
        assert ops.norm_heads(stream, delta, norm_w, EPS, w_qkv, batch, table, cache, **heads, **kinds) is None
        return
    o = ops.paged_attention(q, batch, table, other, **heads, **scores)
    same(got, ops.linear_into_stream(o.view(-1, NQ * HD), w_o, expected, hint), stream, expected)
    assert torch.equal(cache.k_pages, other.k_pages) and torch.equal(cache.v_pages, other.v_pages)


@pytest.mark.parametrize("T", [72, 129, 511, 512, 1000])
def test_feed_forward_in_one_call(gpu_device, T):
    ops = load_hip_ops(gpu_device)
    w_gu, w_down, w_next = ((0.05 * rand(shape, i)).to(gpu_device, torch.bfloat16) for i, shape in enumerate(
        [(2 * INNER, D), (D, INNER), (2048, D)]))
    delta = prepared(gpu_device, T, w_gu, silu_mul=True)
    stream = rand((T, D), 4).to(gpu_device)
    expected = stream.clone()
    hint = NormHint(torch.ones(D, device=gpu_device), EPS, w_next)
    norm_w = delta.hint.norm_weight
    got = ops.feed_into_stream(stream, delta, norm_w, EPS, w_gu, w_down, hint)
    act, _ = ops.norm_linear(expected, delta, norm_w, EPS, w_gu, torch.bfloat16, silu_mul=True)
    same(got, ops.linear_into_stream(act, w_down, expected, hint), stream, expected)
    with pytest.raises(ValueError, match="another norm"):
        ops.feed_into_stream(stream, delta, norm_w.clone(), EPS, w_gu, w_down, hint)
    with pytest.raises(ValueError, match="shape"):
        ops.feed_into_stream(stream[:8], delta, norm_w, EPS, w_gu, w_down, hint)
    small = w_down[:, :512].contiguous()   # (weights whose separate calls stay)
    delta = prepared(gpu_device, T, w_gu[:1024], silu_mul=True)
    assert ops.feed_into_stream(stream, delta, delta.hint.norm_weight, EPS, w_gu[:1024], small, hint) is None
