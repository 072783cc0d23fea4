"""Kernels that keep a row in registers, in fours and an element at a time: rows that end inside a four's
reach, rows longer than the registers, operands that do not begin on 16 bytes."""

import pytest
import torch

from kernel_refs import TorchOps
from test_zonopel_gpu import Scene
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.parts import PagedLatentNeed, SlotStateNeed

pytestmark = pytest.mark.gpu
REF = TorchOps()


def rand(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def placed(x, device, dtype, shifted):
    """x on the device, its first element on 16 bytes or one element behind."""
    room = torch.empty(x.numel() + 8, dtype=dtype, device=device)
    at = 1 if shifted else 0
    out = room[at:at + x.numel()].view(x.shape)
    out.copy_(x)
    return out


def close(got, want, dtype):
    # sums of a row's squares in another order; one rounding to bfloat16
    tol = dict(rtol=2e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(got.float(), want.float(), **tol)


@pytest.mark.parametrize("width", [1, 4, 6, 252, 257, 512, 2044, 2052, 8192, 8196, 8197])
@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows(gpu_device, dtype, shifted, width):
    ops, rows = load_hip_ops(gpu_device), 3

    def f32(seed, shape=(width,), scale=0.1, base=1.0):
        return placed(base + rand(shape, seed, scale), gpu_device, torch.float32, shifted)
    resid, delta = f32(1, (rows, width), 1.0, 0.0), placed(rand((rows, width), 2, 3.0), gpu_device, dtype, shifted)
    other = placed(rand((rows, width), 3), gpu_device, torch.float32, False)
    post, norm = f32(4), f32(5)

    def streams():
        return placed(resid, gpu_device, torch.float32, shifted), resid.clone()
    a, b = streams()
    ops.postnorm_add(a, delta, post, 1e-5)
    REF.postnorm_add(b, delta, post, 1e-5)
    close(a, b, torch.float32)
    a, b = streams()
    close(ops.postnorm_add_norm(a, delta, post, 1e-5, norm, 1e-6, dtype),
          REF.postnorm_add_norm(b, delta, post, 1e-5, norm, 1e-6, dtype), dtype)
    close(a, b, torch.float32)
    for args in ((delta, None, None), (delta, other, None), (delta, other, f32(6))):
        a, b = streams()
        close(ops.stream_add_norm(a, *args, norm, 1e-5, dtype), REF.stream_add_norm(b, *args, norm, 1e-5, dtype),
              dtype)
        close(a, b, torch.float32)
    z = f32(7, (rows, width), 1.0, 0.0)
    coef = torch.tensor([0.3, -0.2, 0.5, 0.1], device=gpu_device)
    close(ops.polynorm(z, coef, 1e-5, dtype), REF.polynorm(z, coef, 1e-5, dtype), dtype)


@pytest.mark.parametrize("width", [1, 4, 6, 252, 2044, 2052, 4100, 16396])
@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embeddings(gpu_device, dtype, shifted, width):
    ops = load_hip_ops(gpu_device)
    table = placed(rand((23, width), 1), gpu_device, dtype, shifted)
    ids = torch.randint(0, 23, (9,), dtype=torch.int32, device=gpu_device)
    assert torch.equal(ops.embed(table, ids), REF.embed(table, ids))
    bigram = placed(rand((12, width), 2), gpu_device, dtype, shifted)
    norm = placed(1 + 0.1 * rand((width,), 3), gpu_device, torch.float32, shifted)
    kw = dict(scale=1.5, buckets=11, mul_prev=31, mul_cur=7, eps=1e-5)
    scene = Scene(gpu_device, SlotStateNeed((1,), torch.int32, "p"), 8, 4)
    mine = scene.view.states["p"]
    mine.fill_(5)
    other = mine.clone()
    for spans in ([3, 1, 2], [1, 1, 1], [1, 4, 1]):       # from the start, then behind tokens
        batch = scene.step(spans)
        batch.token_ids.copy_(torch.randint(0, 23, (batch.num_tokens,), dtype=torch.int32))
        close(ops.bigram_embed(table, bigram, norm, batch, mine, **kw),
              REF.bigram_embed(table, bigram, norm, batch, other, **kw), torch.float32)
        assert torch.equal(mine, other)


@pytest.mark.parametrize("q_rank, kv_rank, rot", [(768, 512, 64), (6, 14, 2), (2052, 2056, 4), (40, 36, 6), (2051, 24, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latent_rows_and_merges(gpu_device, dtype, q_rank, kv_rank, rot):
    ops = load_hip_ops(gpu_device)
    scene = Scene(gpu_device, PagedLatentNeed(kv_rank + rot, None), 16, 2, dtype=dtype, num_pages=40)
    freqs = placed(rand((rot // 2,), 4).abs(), gpu_device, torch.float32, False)
    qn, kn = (placed(1 + 0.1 * rand((n,), s), gpu_device, torch.float32, False)
              for n, s in ((q_rank, 5), (kv_rank, 6)))
    cache, heads = scene.view, 4
    for spans in ([200, 37], [1, 1]):
        batch = scene.step(spans)
        table = batch.tables[0]
        proj = placed(rand((batch.num_tokens, q_rank + kv_rank + rot), 7), gpu_device, torch.float32, False)
        kw = dict(q_rank=q_rank, kv_rank=kv_rank, rot_dim=rot, rot_dims=rot, q_norm=qn, kv_norm=kn, eps=1e-5,
                  freqs=freqs, out_dtype=dtype)
        cache.k_pages.zero_()
        want = REF.latent_prepare(proj, batch, table, cache, **kw)
        pages = cache.k_pages.clone()
        cache.k_pages.zero_()
        close(ops.latent_prepare(proj, batch, table, cache, **kw), want, dtype)
        close(cache.k_pages, pages, dtype)
        cache.k_pages.normal_()
        if kv_rank > 512 or (kv_rank + rot) % 8:
            continue
        qa = rand((batch.num_tokens, heads, kv_rank + rot), 8).to(gpu_device)
        akw = dict(heads=heads, kv_rank=kv_rank, rot_dim=rot, scale=(kv_rank + rot) ** -0.5, window=None,
                   out_dtype=dtype)
        got, want = (o.latent_attention(qa, batch, table, cache, **akw) for o in (ops, REF))
        # (bfloat16 pages go through the matrix cores: queries rounded to 8 bits too)
        tol = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=3e-2, atol=2e-2)
        torch.testing.assert_close(got.float(), want.float(), **tol)
