"""Float32 q, k and v rows on the way to attention: sizes of heads that go eight elements a lane and
one that does not, portions around the 64 tokens from which values are stored tile by tile, pages of
either type, a buffer that does not begin on 16 bytes."""

import dataclasses

import pytest
import torch

from kernel_refs import TorchOps
from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu
REF = TorchOps()


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("pages", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd", [16, 48, 64, 128, 256])
@pytest.mark.parametrize("spans", [[(5, 1)], [(0, 63)], [(3, 64)], [(0, 1), (7, 65), (20, 18)]])
def test_float32_rows(gpu_device, hd, pages, spans, offset):
    ops = load_hip_ops(gpu_device)
    nq, nkv = 4, 2
    batch, cache, table, _ = paged_scenario(gpu_device, pages, nkv=nkv, hd=hd, page_size=16, spans=spans)
    other = dataclasses.replace(cache, k_pages=cache.k_pages.clone(), v_pages=cache.v_pages.clone())
    T, row = batch.num_tokens, (nq + 2 * nkv) * hd
    qkv = torch.empty(T * row + offset, device=gpu_device)[offset:].view(T, row)
    qkv.copy_(rand((T, row), 1))
    angles = 40 * rand((256, hd // 2), 2)
    kw = dict(num_heads=nq, num_kv_heads=nkv, head_dim=hd, q_weight=(1 + 0.1 * rand((hd,), 3)).to(gpu_device),
              k_weight=(1 + 0.1 * rand((hd,), 4)).to(gpu_device), eps=1e-6,
              cos_sin=(angles.cos().to(gpu_device), angles.sin().to(gpu_device)))
    got = ops.qk_norm_rope_store(qkv, batch, table, cache, **kw)
    want = REF.qk_norm_rope_store(qkv, batch, table, other, **kw)
    # float32 throughout: the norm's sum in another order and a dozen roundings; a page of
    # bfloat16 rounds what it is given once (half a unit is 2^-8 of the value)
    torch.testing.assert_close(got, want, rtol=2e-6, atol=4e-6)
    tol = dict(rtol=2e-6, atol=4e-6) if pages == torch.float32 else dict(rtol=2 ** -7, atol=4e-6)
    torch.testing.assert_close(cache.k_pages.float(), other.k_pages.float(), **tol)
    assert torch.equal(cache.v_pages, other.v_pages)          # values are copied
