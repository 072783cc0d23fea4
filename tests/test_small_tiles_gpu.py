"""The tiles of 64 rows of the LDS-tiled product against its others: K is summed in index order by one
accumulator whatever the tile, so every tile gives the same bits, in every form."""

import pytest
import torch

from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.kernels.hip_ops import _ptr
from tokensprint_amd.kernels.stream import NormHint

pytestmark = pytest.mark.gpu
TILES = (6, 7, 8)


def rand(shape, seed, device):
    gen = torch.Generator().manual_seed(seed)
    return (0.1 * torch.randn(shape, generator=gen)).to(device, torch.bfloat16)


@pytest.mark.parametrize("M", [1, 15, 64, 65, 130])
@pytest.mark.parametrize("N, K", [(16, 256), (48, 320), (144, 512), (1344, 256)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_plain_and_paired(gpu_device, out_dtype, M, N, K):
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 1, gpu_device), rand((N, K), 2, gpu_device)
    want = ops.gemm_tiled(x, w, out_dtype, tile=3)
    exact = x.double().cpu() @ w.double().cpu().T
    # K products of 8-bit operands, added in 32 bits; then rounded to the output's type
    tol = 2.0 ** -8 if out_dtype == torch.bfloat16 else K * 2.0 ** -24
    assert (want.double().cpu() - exact).abs().max() <= tol * (x.double().cpu().abs() @ w.double().cpu().abs().T).max()
    for tile in (0,) + TILES:
        assert torch.equal(ops.gemm_tiled(x, w, out_dtype, tile=tile), want), tile
    if out_dtype == torch.bfloat16:
        pair = rand((2 * N, K), 3, gpu_device)
        want = ops.gemm_tiled(x, pair, out_dtype, pair=True, tile=3)
        for tile in (0,) + TILES:
            assert torch.equal(ops.gemm_tiled(x, pair, out_dtype, pair=True, tile=tile), want), tile


@pytest.mark.parametrize("M", [1, 63, 65, 200])
@pytest.mark.parametrize("N, K", [(32, 256), (96, 576), (256, 320)])
def test_tail_and_scaled(gpu_device, M, N, K):
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 1, gpu_device), rand((N, K), 2, gpu_device)
    norm_w = (1 + rand((N,), 3, gpu_device)).float()
    stream = rand((M, N), 4, gpu_device).float()
    parts = ops.lib.ts_gemm_tiled_tail_parts(N)
    results = []
    for tile in (3, 0) + TILES:
        resid, rows = stream.clone(), torch.empty(M, N, device=gpu_device, dtype=torch.bfloat16)
        sums = torch.empty(parts, M, device=gpu_device)
        ops._call(ops.lib.ts_gemm_tiled_tail_bf16, _ptr(x), _ptr(w), _ptr(resid), _ptr(norm_w), _ptr(rows),
                  _ptr(sums), M, N, K, tile, ops._stream())
        results.append((resid, rows, sums))
    assert torch.equal(results[0][0], stream + ops.gemm_tiled(x, w, torch.bfloat16, tile=3).float())
    for got in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got, results[0]))
    if N < 256:
        return
    behind = rand((48, N), 5, gpu_device)
    outs = []
    for tile in (3, 0) + TILES:
        outs.append(torch.empty(M, 48, device=gpu_device))
        ops._call(ops.lib.ts_gemm_tiled_scaled_bf16, _ptr(results[0][1]), _ptr(results[0][2]), parts,
                  _f(1e-6), _ptr(behind), _ptr(outs[-1]), 0, M, 48, N, 0, tile, ops._stream())
    # the same sums with a row's side by side, what is behind the last left as it is
    by_row = torch.full((M, -(-parts // 4) * 4), float("nan"), device=gpu_device)
    by_row[:, :parts] = results[0][2].T
    for pair, out in ((0, torch.empty(M, 48, device=gpu_device)),
                      (1, torch.empty(M, 16, device=gpu_device, dtype=torch.bfloat16))):
        w_behind = behind[:32].contiguous() if pair else behind
        got, want = out.clone(), out
        for name, sums, o in (("ts_gemm_tiled_scaled_rows_bf16", by_row, got),
                              ("ts_gemm_tiled_scaled_bf16", results[0][2], want)):
            ops._call(getattr(ops.lib, name), _ptr(results[0][1]), _ptr(sums), parts, _f(1e-6),
                      _ptr(w_behind), _ptr(o), pair, M, o.shape[1], N, pair, 0, ops._stream())
        assert torch.equal(got, want)


def calls_of(ops, monkeypatch):
    """The names of the library's functions that `ops` calls from now on, in order.  (In the provider's
    own dict, which loses the entry again: all tests share the provider.)"""
    called, call = [], ops._call
    monkeypatch.setitem(vars(ops), "_call", lambda fn, *args: (called.append(fn.__name__), call(fn, *args))[1])
    return called


@pytest.mark.parametrize("M", [16, 17, 32, 33, 64])
@pytest.mark.parametrize("N, silu_mul, rows", [(1040, False, 33), (2048, True, 33), (2064, True, 17)])
@pytest.mark.parametrize("captured", [False, True])
def test_rows_of_the_weight_streaming_tail(gpu_device, monkeypatch, captured, M, N, silu_mul, rows):
    """linear_into_stream and norm_linear at the rows where the second changes its kernel (in steps that
    are captured, or run to be), against float64: two roundings to bfloat16 of operands, and of the results."""
    ops, K, width, eps = load_hip_ops(gpu_device), 2048, 1024, 1e-6
    x, w_o = rand((M, K), 8, gpu_device), rand((width, K), 9, gpu_device)
    resid, norm_w = rand((M, width), 10, gpu_device).float() * 30, (1 + rand((width,), 11, gpu_device)).float()
    weight = rand((N * (2 if silu_mul else 1), width), 12, gpu_device)
    want = resid.double() + (x.double() @ w_o.double().T)
    normed = want / (want.square().mean(-1, keepdim=True) + eps).sqrt() * norm_w.double()
    want_out = normed @ weight.double().T
    if silu_mul:
        want_out = torch.nn.functional.silu(want_out[:, :N]) * want_out[:, N:]
    monkeypatch.setattr(ops, "_timed_plans", captured)
    called = calls_of(ops, monkeypatch)
    prepared = ops.linear_into_stream(x, w_o, resid, NormHint(norm_w, eps, weight, silu_mul))
    assert prepared is not None and not prepared.tiled
    out, _ = ops.norm_linear(resid, prepared, norm_w, eps, weight, torch.bfloat16, silu_mul)
    assert called == ["ts_gemm_tail_bf16", "ts_gemm_tiled_scaled_rows_bf16" if captured and M >= rows
                      else "ts_gemm_scaled_bf16"]
    assert (out.double() - want_out).norm() <= 1e-2 * want_out.norm()


@pytest.mark.parametrize("M", [8, 9, 16, 17, 33, 48, 64])
@pytest.mark.parametrize("N, K", [(16400, 1024), (16400, 2048), (119552, 1088)])
def test_output_heads_of_few_rows(gpu_device, monkeypatch, M, N, K):
    """The weight-streaming kernel's up to 8 rows, the library's from there (which shares K out at up to 16 rows,
    and at some numbers of columns for the last of its tiles): float32 sums of K products."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 6, gpu_device), rand((N, K), 7, gpu_device)
    called = calls_of(ops, monkeypatch)
    out = ops.linear(x, w, torch.float32)
    assert called == ["ts_gemm_mfma_bf16" if M <= 8 else "ts_gemm_library_bf16"]
    exact = x.double() @ w.double().T
    assert (out.double() - exact).norm() <= 4e-6 * exact.norm()
    assert (out.double() - exact).norm() <= 1.02 * (library(ops, x, w).double() - exact).norm()


@pytest.mark.parametrize("M, N, K, tiled", [
    (65, 256, 1024, True), (65, 3072, 1024, True), (65, 3072, 1088, False), (128, 1024, 2048, False),
    (144, 1792, 1088, False), (256, 512, 1536, False), (300, 256, 4096, False), (500, 1024, 1024, True)])
def test_float32_results_of_small_tiles(gpu_device, monkeypatch, M, N, K, tiled):
    """Plain products that leave in float32 are no further from float64 than the library's, which shares K out
    where there are few tiles; in bfloat16 the tiled kernel's in all of these sizes."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 13, gpu_device), rand((N, K), 14, gpu_device)
    exact, called = x.double() @ w.double().T, calls_of(ops, monkeypatch)
    out = ops.linear(x, w, torch.float32)
    ops.linear(x, w, torch.bfloat16)
    error, theirs = ((o.double() - exact).norm() for o in (out, library(ops, x, w)))
    assert error <= 1.05 * theirs
    assert called[:2] == ["ts_gemm_tiled_bf16" if tiled else "ts_gemm_library_bf16", "ts_gemm_tiled_bf16"]


def library(ops, x, w):
    from ctypes import c_size_t
    out, space = torch.empty(x.shape[0], w.shape[0], device=x.device), ops._library_workspace
    ops._call(ops.lib.ts_gemm_library_bf16, _ptr(x), _ptr(w), _ptr(out), 0, x.shape[0], w.shape[0], x.shape[1],
              _ptr(space), c_size_t(space.numel()), ops._stream())
    return out


def _f(value):
    from ctypes import c_float
    return c_float(value)


@pytest.mark.parametrize("T", [32, 33, 64])
def test_prepared_rows_by_kind_of_step(gpu_device, monkeypatch, T):
    """Steps that are captured, or run to be, take the tiled kernel from 33 rows; others do not.  Both sums
    are of the same products, 1,024 of about 0.05 a piece, in bfloat16."""
    ops, K, N = load_hip_ops(gpu_device), 1024, 1536
    x, w, norm_w = (torch.randn(s, generator=torch.Generator().manual_seed(i)).to(gpu_device)
                    for i, s in enumerate([(T, 512), (K, 512), (K,)]))
    w2 = (0.05 * torch.randn(N, K, generator=torch.Generator().manual_seed(4))).to(gpu_device, torch.bfloat16)
    hint, called, results = NormHint(norm_w, 1e-6, w2), calls_of(ops, monkeypatch), []
    for timed in (False, True):
        monkeypatch.setattr(ops, "_timed_plans", timed)
        resid = torch.zeros(T, K, device=gpu_device)
        delta = ops.linear_into_stream(x.bfloat16(), w.bfloat16(), resid, hint)
        results.append(ops.norm_linear(resid, delta, norm_w, 1e-6, w2, torch.bfloat16)[0].float())
    captured = "ts_gemm_tiled_scaled_rows_bf16" if T >= 33 else "ts_gemm_scaled_bf16"
    assert called == ["ts_gemm_tail_bf16", "ts_gemm_scaled_bf16", "ts_gemm_tail_bf16", captured]
    # float32 sums of 1,024 terms in two orders, then one rounding to bfloat16 each
    assert (results[0] - results[1]).abs().max() <= 2 ** -7 * results[0].abs().max()


@pytest.mark.parametrize("T", [17, 33, 64])
def test_float32_rows_are_the_same_in_both_kinds_of_step(gpu_device, monkeypatch, T):
    """Float32 results keep the weight-streaming kernel, whose sums round less (a third at K = 1,024)."""
    ops, K, N = load_hip_ops(gpu_device), 1024, 1536
    x, w, resid = (torch.randn(s, generator=torch.Generator().manual_seed(i)).to(gpu_device)
                   for i, s in enumerate([(T, 512), (K, 512), (T, K)]))
    w2, ones = rand((N, K), 4, gpu_device), torch.ones(K, device=gpu_device)
    hint, called, results = NormHint(ones, 1e-6, w2), calls_of(ops, monkeypatch), []
    for captured in (False, True):
        monkeypatch.setattr(ops, "_timed_plans", captured)
        stream = resid.clone()
        prepared = ops.linear_into_stream(x.bfloat16(), w.bfloat16(), stream, hint)
        results.append(ops.norm_linear(stream, prepared, ones, 1e-6, w2, torch.float32)[0])
    assert called == ["ts_gemm_tail_bf16", "ts_gemm_scaled_bf16"] * 2
    assert torch.equal(*results)
