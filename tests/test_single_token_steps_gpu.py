"""Kernels of steps in which every entry brings one token against the ones that take entries of
any length, at the edges of their sizes.  They add the same sums in the same order, so outputs
and the states that are left are equal to the bit (operands that do not begin on 16 bytes go to
the general kernels)."""

import pytest
import torch

from tokensprint_amd.cache import CacheManager, CacheStorage
from tokensprint_amd.engine.batch import BatchBuilder, StepEntry
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.parts.base import SlotStateNeed

pytestmark = pytest.mark.gpu


def rand(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).cuda()


def steps(device, entries, count):
    """`count` steps of one token an entry; slots do not start at 0."""
    storage = CacheStorage([SlotStateNeed((1,), torch.float32, "s")], 16, 8, entries + 2,
                           torch.float32, device)
    manager = CacheManager(storage.groups, 16, 8, entries + 2)
    manager.admit("in front")
    caches = [manager.admit(i) for i in range(entries)]
    builder = BatchBuilder(device, len(storage.groups))
    for _ in range(count):
        out = []
        for rc in caches:
            manager.extend(rc, rc.num_tokens + 1)
            out.append(StepEntry(rc, [1], rc.num_tokens - 1, [0]))
        yield builder.build(out)


def off_by_one(t):
    """A copy of t that begins 4 bytes behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + 4, dtype=t.dtype, device=t.device)
    view = buf[1:1 + t.numel()].view(t.shape)
    view.copy_(t)
    return view


def stale(entries, shape):
    """What others left in the slots: not numbers, which a new sequence must not see."""
    return torch.full((entries + 2, *shape), float("nan"), device="cuda")


@pytest.mark.parametrize("form", ["fixed", "silu", "turn", "per_head", "delta", "per_row"])
@pytest.mark.parametrize("heads, kv_heads, N, P, entries", [
    (2, 1, 16, 4, 1), (4, 2, 32, 60, 3), (2, 2, 64, 64, 2), (3, 1, 64, 68, 5), (4, 2, 128, 128, 2),
    (2, 1, 128, 132, 1), (2, 2, 24, 64, 2)])
def test_recurrence(gpu_device, form, heads, kv_heads, N, P, entries):
    ops = load_hip_ops(gpu_device)
    if form in ("fixed", "silu", "turn"):
        kv_heads = heads
    qk = kv_heads * N
    kw = dict(heads=heads, kv_heads=kv_heads, dim=N, vdim=P, silu_inputs=form == "silu")
    if form in ("fixed", "silu", "turn"):
        kw["decay"] = torch.rand(heads, generator=torch.Generator().manual_seed(1)).cuda()
    if form == "turn":
        kw.update(turn=rand((8, N // 2 - 2, 2), 2), k_scale=0.3)
    one, other = stale(entries, (heads, N, P)), stale(entries, (heads, N, P))
    other = off_by_one(other)
    for i, batch in enumerate(steps(gpu_device, entries, 3)):
        x = rand((entries, 4 + 2 * qk + heads * P), 10 + i, 0.5)
        if form in ("per_head", "delta", "per_row"):
            n = heads * N if form == "per_row" else heads
            kw.update(gates=torch.sigmoid(rand((entries, heads + n), 20 + i)),
                      delta=form != "per_head", per_channel=form == "per_row")
        got = ops.linear_recurrence(x, 4, 4 + qk, 4 + 2 * qk, batch, one, **kw)
        want = ops.linear_recurrence(x, 4, 4 + qk, 4 + 2 * qk, batch, other, **kw)
        assert not got.isnan().any()
        assert torch.equal(got, want) and torch.equal(one[1:-1], other[1:-1])


@pytest.mark.parametrize("heads, groups, N, P, entries", [
    (2, 1, 16, 4, 1), (4, 2, 32, 60, 3), (4, 4, 64, 64, 2), (8, 2, 128, 64, 5), (2, 1, 128, 68, 2),
    (2, 1, 24, 64, 2)])
def test_state_space(gpu_device, heads, groups, N, P, entries):
    ops = load_hip_ops(gpu_device)
    args = [rand((heads,), 1), rand((heads,), 2), rand((heads,), 3)]
    kw = dict(heads=heads, vdim=P, state_rows=N, groups=groups)
    one = stale(entries, (heads, N, P))
    other = off_by_one(one)
    for i, batch in enumerate(steps(gpu_device, entries, 3)):
        xbc = rand((entries, heads * P + 2 * groups * N), 10 + i)
        proj = rand((entries, 3 + heads), 20 + i)
        got = ops.ssm_scan(xbc, proj, 3, *args, batch, one, **kw)
        want = ops.ssm_scan(xbc, proj, 3, *args, batch, other, **kw)
        assert not got.isnan().any()
        assert torch.equal(got, want) and torch.equal(one[1:-1], other[1:-1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("heads, kv_heads, N, P, entries", [
    (2, 1, 16, 64, 1), (4, 2, 32, 128, 3), (2, 2, 64, 64, 2), (6, 2, 128, 128, 5)])
def test_delta_rule_whole(gpu_device, heads, kv_heads, N, P, entries, per_channel, dtype):
    """From the convolved rows to the gated ones against the three kernels one after the other."""
    ops = load_hip_ops(gpu_device)
    qk, inner, n = kv_heads * N, heads * P, heads * N if per_channel else heads
    a_log, dt_bias, w = rand((heads,), 1), rand((n,), 2), 1 + 0.1 * rand((P,), 3)
    one, other = stale(entries, (heads, N, P)), stale(entries, (heads, N, P))
    sizes = dict(heads=heads, kv_heads=kv_heads, dim=N)
    out = dict(gate="sigmoid" if per_channel else "silu", eps=1e-6, out_dtype=dtype)
    for i, batch in enumerate(steps(gpu_device, entries, 3)):
        qkv, proj = rand((entries, 2 * qk + inner), 10 + i), rand((entries, 5 + heads), 20 + i)
        z, gate = rand((entries, 3 + n), 30 + i), rand((entries, 8 + inner), 40 + i)
        kept = qkv.clone()
        got = ops.delta_step(qkv, proj, 5, z, 3, a_log, dt_bias, gate, 8, w, batch, one,
                             per_channel=per_channel, vdim=P, **sizes, **out)
        assert torch.equal(qkv, kept)
        gates = ops.delta_gates(qkv, proj, 5, z, 3, a_log, dt_bias, per_channel=per_channel, **sizes)
        o = ops.linear_recurrence(qkv, 0, qk, 2 * qk, batch, other, vdim=P, silu_inputs=False,
                                  gates=gates, per_channel=per_channel, delta=True, **sizes)
        want = ops.norm_gate(o, gate, 8, w, groups=heads, **out)
        assert not got.isnan().any()
        assert torch.equal(got, want) and torch.equal(one[1:-1], other[1:-1])
        # rows that the kernel does not take are left to the others
        assert ops.delta_step(qkv, proj, 5, z, 3, a_log, dt_bias, gate, 7, w, batch, one,
                              per_channel=per_channel, vdim=P, **sizes, **out) is None


@pytest.mark.parametrize("bias, in_bias, plain", [(True, False, False), (False, True, True),
                                                  (False, False, False)])
@pytest.mark.parametrize("entries", [1, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("N, K, col, channels", [(3088, 512, 4, 3084), (1100, 1096, 20, 64),
                                                 (2500, 2048, 0, 2500), (1040, 2056, 1036, 4)])
def test_product_and_convolution(gpu_device, N, K, col, channels, entries, bias, in_bias, plain):
    ops = load_hip_ops(gpu_device)
    weight = (rand((N, K), 1) * K ** -0.5).bfloat16()
    conv_w = rand((channels, 4), 2)
    b = rand((channels,), 3) if bias else None
    ib = rand((channels,), 4) if in_bias else None
    one, other = stale(entries, (3, channels)), stale(entries, (3, channels))
    for i, batch in enumerate(steps(gpu_device, entries, 5)):
        x = rand((entries, K), 10 + i).bfloat16()
        proj, got = ops.linear_conv_silu(x, weight, col, channels, conv_w, b, batch, one,
                                         in_bias=ib, plain=plain)
        rows = ops.linear(x, weight, torch.float32)
        want = ops.conv_silu(rows, col, channels, conv_w, b, batch, other, in_bias=ib, plain=plain)
        assert not got.isnan().any()
        assert torch.equal(proj, rows) and torch.equal(got, want)
        assert torch.equal(one[1:-1], other[1:-1])


@pytest.mark.parametrize("delta_type", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width, entries", [(4, 1), (100, 3), (2048, 8), (8192, 2), (8200, 2)])
def test_add_norm_and_shift(gpu_device, width, entries, delta_type):
    ops = load_hip_ops(gpu_device)
    post, norm, shift = (1 + 0.1 * rand((width,), s) for s in (1, 2, 3))
    one, other = stale(entries, (width,)), stale(entries, (width,))
    for i, batch in enumerate(steps(gpu_device, entries, 3)):
        a, delta = rand((entries, width), 10 + i), rand((entries, width), 20 + i).to(delta_type)
        b = a.clone()
        got = ops.postnorm_add_shift(a, delta, post, 1e-5, norm, 1e-6, shift, batch, one,
                                     torch.bfloat16)
        ops.postnorm_add(b, delta, post, 1e-5)
        want = ops.norm_token_shift(b, norm, 1e-6, shift, batch, other, torch.bfloat16)
        assert not got.isnan().any()
        assert torch.equal(a, b) and torch.equal(got, want) and torch.equal(one[1:-1], other[1:-1])


@pytest.mark.parametrize("T, n_a, k_a, n_g, k_g, col", [(1, 16, 32, 16, 32, 0), (8, 512, 64, 1024, 64, 8),
                                                        (17, 70, 96, 5, 64, 3), (300, 512, 64, 1000, 32, 4)])
def test_low_rank_pair(T, n_a, k_a, n_g, k_g, col):
    """Two products over columns of float32 rows (also where they do not begin on 16 bytes) against
    copies of the columns and products of their own."""
    ops = load_hip_ops("cuda:0")
    ld = col + k_a + k_g + 3
    x = rand((T, ld), 90)
    w_a, w_g = (rand((n, k), 91, 0.1).to(torch.bfloat16) for n, k in ((n_a, k_a), (n_g, k_g)))
    z, gate = ops.low_rank_pair(x, col, w_a, col + k_a, w_g, torch.bfloat16)
    for got, at, w in ((z, col, w_a), (gate, col + k_a, w_g)):
        want = x[:, at:at + w.shape[1]].to(torch.bfloat16).double() @ w.double().T
        # float32 sums of K exact products: K roundings at most of partial sums below |x| |w|
        bound = x[:, at:at + w.shape[1]].abs().double() @ w.abs().double().T * w.shape[1] * 2.0 ** -24
        assert ((got.double() - want).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize("T, n_a, k_a, n_g, k_g, one", [
    (2048, 512, 64, 1024, 64, True), (2049, 512, 64, 1024, 64, False), (8, 64, 512, 64, 512, True),
    (8, 64, 544, 64, 512, False), (200, 4096, 512, 4096, 512, False)])
def test_low_rank_pairs_that_are_two_products(monkeypatch, T, n_a, k_a, n_g, k_g, one):
    """Long ranks and many rows are left to the products of their own, which share operands out."""
    ops = load_hip_ops("cuda:0")
    taken, linear = [], ops.linear
    monkeypatch.setitem(vars(ops), "linear", lambda x, w, t: taken.append(w) or linear(x, w, t))
    x = rand((T, k_a + k_g), 92)
    w_a, w_g = (rand((n, k), 93, 0.1).to(torch.bfloat16) for n, k in ((n_a, k_a), (n_g, k_g)))
    z, gate = ops.low_rank_pair(x, 0, w_a, k_a, w_g, torch.bfloat16)
    assert len(taken) == (0 if one else 2)
    for got, at, w in ((z, 0, w_a), (gate, k_a, w_g)):
        want = x[:, at:at + w.shape[1]].to(torch.bfloat16).float() @ w.float().T
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-3)
