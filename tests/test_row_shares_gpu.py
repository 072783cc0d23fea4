"""Kernels that keep a row in registers, in fours and an element at a time: rows that end inside a four's
reach, rows longer than the registers, operands that do not begin on 16 bytes."""

import pytest
import torch

from kernel_refs import TorchOps
from tokensprint_amd.kernels import load_hip_ops

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
