"""Parts of rows normed and gated, and the short convolution four channels a thread, at the sizes
where a kernel takes over from the next, against their torch twins."""

import pytest
import torch

from kernel_refs import TorchOps
from tokensprint_amd.cache import CacheManager, CacheStorage
from tokensprint_amd.engine.batch import BatchBuilder, StepEntry
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.parts.base import SlotStateNeed

pytestmark = pytest.mark.gpu
REF = TorchOps()


def rand(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("size", [4, 64, 68, 128, 132, 256, 260, 512, 516, 1024, 1028, 2048, 2052, 4096, 4100])
def test_parts_normed_and_gated(gpu_device, size, dtype):
    ops = load_hip_ops(gpu_device)
    # one rounding of the result, and a few float32 units in front of it
    tol = dict(rtol=2e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=8e-3, atol=1e-5)
    for T, groups in ((1, 1), (7, 3), (33, 2)):
        inner = groups * size
        y = rand((T, inner), 1, 3.0).to(gpu_device)
        gate = rand((T, inner + 8), 2).to(gpu_device)
        for w in (None, 1 + 0.1 * rand((size,), 3), 1 + 0.1 * rand((inner,), 4)):
            w = None if w is None else w.to(gpu_device)
            for kind, col in (("sigmoid", 8), ("silu", 4), ("silu", 3)):
                kw = dict(groups=groups, gate=kind, eps=1e-5, out_dtype=dtype)
                torch.testing.assert_close(ops.norm_gate(y, gate, col, w, **kw),
                                           REF.norm_gate(y, gate, col, w, **kw), **tol)
        w = (1 + 0.1 * rand((inner,), 5)).to(gpu_device)
        torch.testing.assert_close(ops.gated_group_norm(y, gate, w, groups, 1e-5, dtype),
                                   REF.gated_group_norm(y, gate, w, groups, 1e-5, dtype), **tol)


@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("channels, ld, col", [(4, 8, 4), (1028, 1040, 8), (64, 67, 0)])
def test_convolution_of_long_steps(gpu_device, channels, ld, col, taps):
    ops = load_hip_ops(gpu_device)
    storage = CacheStorage([SlotStateNeed((taps - 1, channels), torch.float32, "c")], 16, 8, 6,
                           torch.float32, gpu_device)
    manager = CacheManager(storage.groups, 16, 8, 6)
    caches = [manager.admit(i) for i in range(5)]
    builder = BatchBuilder(gpu_device, len(storage.groups))
    state = storage.views[0].states["c"]
    state.fill_(5.0)
    twin = state.clone()
    w, bias = rand((channels, taps), 1).to(gpu_device), rand((channels,), 2).to(gpu_device)
    in_bias = rand((channels,), 3).to(gpu_device)
    for step, spans in enumerate(([270, 1, 2, 9, 16], [1, 300, 8, 1, 3])):
        entries = []
        for rc, n in zip(caches, spans):
            manager.extend(rc, rc.num_tokens + n)
            entries.append(StepEntry(rc, [1] * n, rc.num_tokens - n, [n - 1]))
        batch = builder.build(entries)
        x = rand((batch.num_tokens, ld), 10 + step).to(gpu_device)
        for args in (dict(), dict(in_bias=in_bias, plain=True)):
            a, b = state.clone(), twin.clone()
            got = ops.conv_silu(x, col, channels, w, bias, batch, a, **args)
            want = REF.conv_silu(x, col, channels, w, bias, batch, b, **args)
            torch.testing.assert_close(got, want, rtol=2e-5, atol=2e-5)
            torch.testing.assert_close(a, b, rtol=2e-5, atol=2e-5)
        state.copy_(a)
        twin.copy_(b)
