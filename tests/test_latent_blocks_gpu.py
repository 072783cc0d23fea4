"""Latent attention of many tiles: every size that has a kernel of its own, rows shorter than
one, windows and portions that begin and end inside a block of keys, against float32 torch."""

import dataclasses

import pytest
import torch

from tokensprint_amd.cache import CacheManager, CacheStorage
from tokensprint_amd.engine.batch import BatchBuilder, StaticDecodeBatch, StepEntry
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.parts.base import PagedLatentNeed

pytestmark = pytest.mark.gpu


def rand(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("window", [None, 1, 63, 65, 130])
@pytest.mark.parametrize("heads, kv_rank, rot_dim", [
    (3, 64, 32), (5, 128, 32), (4, 256, 32), (2, 256, 64), (16, 512, 64),
    (3, 48, 24), (2, 96, 32), (7, 200, 16), (2, 448, 64), (3, 512, 128)])
def test_tiles_of_one_entry_walk_their_keys_together(gpu_device, monkeypatch, heads, kv_rank,
                                                     rot_dim, window, out_dtype):
    ops = load_hip_ops(gpu_device)
    monkeypatch.setattr(ops, "dispatch", dataclasses.replace(ops.dispatch, latent_full_tiles=1))
    dl, page = kv_rank + rot_dim, 16
    scale = 2.0 / dl ** 0.5
    storage = CacheStorage([PagedLatentNeed(dl, None)], page, 40, 3, torch.bfloat16, gpu_device)
    manager = CacheManager(storage.groups, page, 40, 3)
    builder = BatchBuilder(gpu_device, len(storage.groups))
    view = storage.views[0]
    view.k_pages.copy_(rand(view.k_pages.shape, 1).to(gpu_device).bfloat16())
    caches, at = [manager.admit(i) for i in range(3)], [0, 0, 0]
    sink = rand((heads,), 2).to(gpu_device)
    for spans in ([63, 1, 17], [2, 64, 47], [66, 65, 1]):
        entries = []
        for i, n in enumerate(spans):
            manager.extend(caches[i], at[i] + n)
            entries.append(StepEntry(caches[i], [1] * n, at[i], [n - 1]))
            at[i] += n
        batch = builder.build(entries)
        T = batch.num_tokens
        rows = rand((T, heads * dl), 3, 1.5).to(gpu_device)
        got = ops.latent_attention(rows, batch, batch.tables[0], view, heads=heads, kv_rank=kv_rank,
                                   rot_dim=rot_dim, scale=scale, window=window, sink=sink,
                                   out_dtype=out_dtype).float().view(T, heads, kv_rank)
        row = 0
        for b, e in enumerate(entries):
            keys = torch.arange(e.start + len(e.tokens), device=gpu_device)
            kv = view.k_pages[batch.tables[0][b, keys // page].long(), keys % page].float()
            for i in range(len(e.tokens)):
                p = e.start + i
                lo = 0 if window is None else max(0, p - window + 1)
                mine = kv[lo:p + 1]
                q = rows[row].view(heads, dl).bfloat16().float()
                w = torch.softmax(torch.cat([(mine @ q.T) * scale, sink.view(1, -1)]), 0)[:-1]
                want = w.T @ mine[:, :kv_rank]
                # each weight is rounded to bfloat16 once (8 significant bits: half a unit is 2^-8
                # of the value), and the result where it is bfloat16
                bound = 2 ** -8 * (w.T @ mine[:, :kv_rank].abs()) + 1e-4
                if out_dtype == torch.bfloat16:
                    bound = bound + 2 ** -8 * (want.abs() + bound)
                assert bool(((got[row] - want).abs() <= bound).all()), (spans, b, i)
                row += 1



@pytest.mark.parametrize("heads, kv_rank, rot_dim", [(16, 512, 64), (5, 128, 32), (16, 448, 64),
                                                     (3, 512, 128)])
def test_lanes_without_pages_read_none(gpu_device, monkeypatch, heads, kv_rank, rot_dim):
    """A captured decode step's idle lanes: position 0, no pages.  Their rows see nothing but
    zeros, and the lanes beside them what the form for few tiles gives."""
    ops = load_hip_ops(gpu_device)
    dl, page = kv_rank + rot_dim, 16
    # (the second of two runs: a page in front of its first is the first run's last)
    storage = CacheStorage([PagedLatentNeed(dl, None)] * 2, page, 12, 3, torch.bfloat16, gpu_device)
    manager = CacheManager(storage.groups, page, 12, 3)
    for i, view in enumerate(storage.views):
        view.k_pages.copy_(rand(view.k_pages.shape, 4 + i).to(gpu_device).bfloat16())
    view = storage.views[1]
    entries = []
    for i, n in enumerate((70, 1, 33)):
        cache = manager.admit(i)
        manager.extend(cache, n)
        entries.append(StepEntry(cache, [1], n - 1, [0]))
    static = StaticDecodeBatch(gpu_device, 6, [8], idle_slot=storage.idle_slot)
    static.batch.max_ctx_len = 128
    static.fill(entries)
    rows = rand((6, heads * dl), 6, 1.5).to(gpu_device)
    kept, outs = ops.dispatch, []
    for full in (1, 1 << 30):
        monkeypatch.setattr(ops, "dispatch", dataclasses.replace(kept, latent_full_tiles=full))
        outs.append(ops.latent_attention(
            rows, static.batch, static.batch.tables[0], view, heads=heads, kv_rank=kv_rank,
            rot_dim=rot_dim, scale=2.0 / dl ** 0.5, window=None))
    assert (outs[0][3:] == 0).all() and (outs[1][3:] == 0).all()
    # a weight is rounded to bfloat16 once in either form, 2^-8 of it: the values are up to 5
    assert ((outs[0] - outs[1]).abs() <= 2 * 2 ** -8 * 5).all()
    assert (outs[0][:3] != 0).any(dim=(1, 2)).all()


@pytest.mark.parametrize("window", [None, 37, 64, 100])
@pytest.mark.parametrize("heads, kv_rank, rot_dim", [(16, 512, 64), (2, 128, 32), (5, 200, 16),
                                                     (16, 512, 128)])
def test_rows_do_not_depend_on_how_a_prompt_is_cut(gpu_device, monkeypatch, heads, kv_rank, rot_dim,
                                                   window):
    """Which tokens share a workgroup decides nothing: blocks of keys lie at fixed positions."""
    ops = load_hip_ops(gpu_device)
    monkeypatch.setattr(ops, "dispatch", dataclasses.replace(ops.dispatch, latent_full_tiles=1))
    dl, page, T = kv_rank + rot_dim, 16, 300
    rows = rand((T, heads * dl), 7, 1.5).to(gpu_device)

    def whole(portions):
        storage = CacheStorage([PagedLatentNeed(dl, None)], page, 20, 1, torch.bfloat16, gpu_device)
        manager = CacheManager(storage.groups, page, 20, 1)
        builder, view = BatchBuilder(gpu_device, len(storage.groups)), storage.views[0]
        view.k_pages.copy_(rand(view.k_pages.shape, 8).to(gpu_device).bfloat16())
        cache, at, outs = manager.admit(0), 0, []
        for n in portions:
            manager.extend(cache, at + n)
            batch = builder.build([StepEntry(cache, [1] * n, at, [n - 1])])
            outs.append(ops.latent_attention(
                rows[at:at + n].contiguous(), batch, batch.tables[0], view, heads=heads,
                kv_rank=kv_rank, rot_dim=rot_dim, scale=2.0 / dl ** 0.5, window=window))
            at += n
        assert at == T
        return torch.cat(outs)

    want = whole([T])
    for portions in ([33, 67, 200], [1, 2, 3, 93, 1, 95, 105], [131, 169]):
        assert torch.equal(whole(portions), want), portions
