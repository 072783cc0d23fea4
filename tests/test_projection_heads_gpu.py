"""The q/k/v projection of prepared rows with the heads' preparation in its epilogue, against the product
and the preparation kernel one after the other: the same sums in the same order, so the same bits."""

import dataclasses

import pytest
import torch

from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.kernels.stream import NormHint, PreparedRows

pytestmark = pytest.mark.gpu
#: portions (start, tokens): a tile's edges, runs of sixteen places that begin inside a page, requests
#: that end inside a run, single tokens
SPANS = [[(0, 72)], [(0, 128)], [(0, 257)], [(3, 129), (0, 1), (100, 60)], [(16, 40), (777, 300), (5, 1), (8, 16)]]


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("spans", SPANS)
@pytest.mark.parametrize("page", [16, 64, 4])
@pytest.mark.parametrize("nq, nkv, K, normed, turned, tile", [
    (4, 2, 256, True, True, 1), (4, 2, 256, True, True, 2), (5, 1, 512, False, True, 1),
    (3, 3, 320, True, False, 2), (4, 2, 256, True, True, 6), (2, 1, 512, True, True, 6)])
def test_same_bits_as_the_kernels_one_by_one(gpu_device, nq, nkv, K, normed, turned, tile, page, spans):
    ops, hd, eps = load_hip_ops(gpu_device), 128, 1e-6
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=nkv, hd=hd, page_size=page,
                                            spans=spans)
    other = dataclasses.replace(cache, k_pages=cache.k_pages.clone(), v_pages=cache.v_pages.clone())
    T, N = batch.num_tokens, (nq + 2 * nkv) * hd
    weight = (0.05 * rand((N, K), 1)).to(gpu_device, torch.bfloat16)
    norm_w = torch.ones(K, device=gpu_device)
    rows = rand((T, K), 2).to(gpu_device, torch.bfloat16)
    sumsq = (rand((K // 32, T), 3).square() * 20 + 1).to(gpu_device)
    hint = NormHint(norm_w, eps, weight)
    delta = PreparedRows(rows, sumsq, K // 32, hint, tiled=True)
    resid = torch.zeros(T, K, device=gpu_device)
    angles = 40 * rand((1200, hd // 2), 4)
    q_w, k_w = ((1 + 0.1 * rand((hd,), i)).to(gpu_device) if normed else None for i in (5, 6))
    cos_sin = (angles.cos().to(gpu_device), angles.sin().to(gpu_device)) if turned else None
    got = ops.norm_heads(resid, delta, norm_w, eps, weight, batch, table, cache, num_heads=nq,
                         num_kv_heads=nkv, head_dim=hd, q_weight=q_w, k_weight=k_w, head_eps=1e-5,
                         cos_sin=cos_sin, tile=tile)
    qkv, _ = ops.norm_linear(resid, delta, norm_w, eps, weight, torch.bfloat16)
    want = ops.qk_norm_rope_store(qkv, batch, table, other, num_heads=nq, num_kv_heads=nkv, head_dim=hd,
                                  q_weight=q_w, k_weight=k_w, eps=1e-5, cos_sin=cos_sin)
    assert torch.equal(got, want)
    assert torch.equal(cache.k_pages, other.k_pages)
    assert torch.equal(cache.v_pages, other.v_pages)


def test_rows_of_another_norm_are_refused(gpu_device):
    ops = load_hip_ops(gpu_device)
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=2, hd=128, page_size=16,
                                            spans=[(0, 512)])
    weight = torch.zeros(1024, 256, device=gpu_device, dtype=torch.bfloat16)
    norm_w = torch.ones(256, device=gpu_device)
    delta = PreparedRows(torch.zeros(512, 256, device=gpu_device, dtype=torch.bfloat16),
                         torch.ones(8, 512, device=gpu_device), 8, NormHint(norm_w, 1e-6, weight), tiled=True)
    kw = dict(num_heads=4, num_kv_heads=2, head_dim=128, q_weight=None, k_weight=None, head_eps=1e-6,
              cos_sin=None, tile=2)
    resid = torch.zeros(512, 256, device=gpu_device)
    with pytest.raises(ValueError, match="another norm"):
        ops.norm_heads(resid, delta, norm_w.clone(), 1e-6, weight, batch, table, cache, **kw)
    with pytest.raises(ValueError, match="shape"):
        ops.norm_heads(resid[:8], delta, norm_w, 1e-6, weight, batch, table, cache, **kw)
    kw["head_dim"] = 64
    assert ops.norm_heads(resid, delta, norm_w, 1e-6, weight, batch, table, cache, **kw) is None
