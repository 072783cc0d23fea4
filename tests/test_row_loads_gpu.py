"""Kernels that ask for all of a thread's share at once and drop what does not exist: rows that end inside a
thread's share, taps beyond a four, weights that do not begin on 16 bytes."""

import pytest
import torch

from kernel_refs import TorchOps
from test_row_parts_gpu import rand
from tokensprint_amd.cache import CacheManager, CacheStorage
from tokensprint_amd.engine.batch import BatchBuilder, StepEntry
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.parts.base import SlotStateNeed

pytestmark = pytest.mark.gpu
REF = TorchOps()


@pytest.mark.parametrize("width", [4, 252, 1020, 1028, 2044, 2052, 4092, 4100, 5120, 8188, 8192, 8196])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norms_of_rows(gpu_device, dtype, width):
    ops = load_hip_ops(gpu_device)
    resid, delta = rand((3, width), 1).to(gpu_device), rand((3, width), 2).to(gpu_device, dtype)
    w = (1 + 0.1 * rand((width,), 3)).to(gpu_device)
    # sums of a row's squares in another order; one rounding to bfloat16
    tol = dict(rtol=2e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(ops.rmsnorm(resid, w, 1e-5, dtype), REF.rmsnorm(resid, w, 1e-5, dtype), **tol)
    twin = resid.clone()
    got, want = ops.add_rmsnorm(resid, delta, w, 1e-5, dtype), REF.add_rmsnorm(twin, delta, w, 1e-5, dtype)
    assert torch.equal(resid, twin)
    torch.testing.assert_close(got, want, **tol)


@pytest.mark.parametrize("taps", [2, 3, 4, 5, 6, 8, 9])
@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("bias", [False, True])
def test_convolution_taps(gpu_device, taps, shifted, bias):
    ops, channels = load_hip_ops(gpu_device), 36
    storage = CacheStorage([SlotStateNeed((taps - 1, channels), torch.float32, "c")], 16, 8, 6,
                           torch.float32, gpu_device)
    manager, builder = CacheManager(storage.groups, 16, 8, 6), BatchBuilder(gpu_device, len(storage.groups))
    caches, state = [manager.admit(i) for i in range(4)], storage.views[0].states["c"]
    state.fill_(5.0)
    twin = state.clone()
    room = torch.empty(channels * taps + 4, device=gpu_device)
    w = room[shifted:shifted + channels * taps].view(channels, taps)
    w.copy_(rand((channels, taps), 1))
    b = rand((channels,), 2).to(gpu_device) if bias else None
    for step, spans in enumerate(([1, 257, 2, 5], [3, 1, 260, 7])):
        entries = []
        for rc, n in zip(caches, spans):
            manager.extend(rc, rc.num_tokens + n)
            entries.append(StepEntry(rc, [1] * n, rc.num_tokens - n, [n - 1]))
        batch = builder.build(entries)
        x = rand((batch.num_tokens, channels + 8), 10 + step).to(gpu_device)
        got = ops.conv_silu(x, 4, channels, w, b, batch, state)
        want = REF.conv_silu(x, 4, channels, w, b, batch, twin)
        torch.testing.assert_close(got, want, rtol=2e-5, atol=2e-5)
        assert torch.equal(state, twin)
