"""The recurrences in chunks (chunked_state.hip) against a token-by-token walk in float64, at the
edges of their tiles and chunks: errors are held to those of the kernels that walk in float32."""

import dataclasses

import pytest
import torch

from tokensprint_amd.cache import CacheManager, CacheStorage
from tokensprint_amd.engine.batch import BatchBuilder, StepEntry
from tokensprint_amd.kernels import load_hip_ops
from tokensprint_amd.kernels.hip_ops import KernelError
from tokensprint_amd.parts.base import SlotStateNeed

pytestmark = pytest.mark.gpu


def walk(q, k, v, g, beta, S):
    """q, k [T, H, N], v [T, H, P], g [T, H, N or 1], beta [T, H] or None, S [H, N, P], float64."""
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = S * g[t].unsqueeze(-1)
        u = v[t] if beta is None else beta[t, :, None] * (v[t] - (S * k[t].unsqueeze(-1)).sum(1))
        S = S + k[t].unsqueeze(-1) * u.unsqueeze(1)
        out[t] = (S * q[t].unsqueeze(-1)).sum(1)
    return out, S


class Requests:
    def __init__(self, device, shape, count):
        self.storage = CacheStorage([SlotStateNeed(shape, torch.float32, "s")], 16, 8, count + 2,
                                    torch.float32, device)
        self.manager = CacheManager(self.storage.groups, 16, 8, count + 2)
        self.manager.admit("in front")                     # so that slots do not start at 0
        self.caches = [self.manager.admit(i) for i in range(count)]
        self.builder = BatchBuilder(device, len(self.storage.groups))
        self.state = self.storage.views[0].states["s"]
        self.state.fill_(3.0)                              # what others left in the slots

    def step(self, spans):
        entries = []
        for rc, n in zip(self.caches, spans):
            self.manager.extend(rc, rc.num_tokens + n)
            entries.append(StepEntry(rc, [1] * n, rc.num_tokens - n, [n - 1]))
        return self.builder.build(entries)


def in_chunks_and_walked(ops, call, state):
    """`call`'s output and the state it leaves, by the chunked kernels and by those that walk."""
    before, kept = state.clone(), ops.dispatch
    results = []
    try:
        for whole in (16, 1 << 30):
            ops.dispatch = dataclasses.replace(kept, scan_whole_tokens=whole,
                                               state_space_whole_tokens=whole)
            state.copy_(before)
            results.append((call(), state.clone()))
    finally:
        ops.dispatch = kept
    state.copy_(results[0][1])
    return results


def no_further_off(chunked, walked, want):
    """Both are float32 sums of the same products, in other orders: what the walk is off by is what
    the sizes and the data give, and a few units in the last place of the largest value."""
    scale = want.abs().max().item()
    off = [(x.double().cpu() - want).norm().item() / max(want.norm().item(), 1e-30)
           for x in (chunked, walked)]
    top = (chunked.double().cpu() - want).abs().max().item()
    assert off[0] <= 2 * off[1] + 1e-6, off
    assert top <= 1e-4 * scale, (top, scale)


SPANS = [[130, 1, 64, 17], [1, 65, 3, 200]]
SIZES = [(4, 2, 128, 128), (2, 2, 64, 64), (3, 1, 10, 6), (2, 1, 36, 70), (1, 1, 65, 17)]


@pytest.mark.parametrize("mode", ["fixed", "per_head_plain", "turned", "delta", "delta_per_channel"])
@pytest.mark.parametrize("heads, kv_heads, dim, vdim", SIZES + [(2, 2, 200, 33)])
def test_linear_recurrence_in_chunks(gpu_device, mode, heads, kv_heads, dim, vdim):
    if dim > 128 and mode.startswith("delta"):
        pytest.skip("the delta rule runs in chunks up to 128 rows")
    ops = load_hip_ops(gpu_device)
    qk, inner = kv_heads * dim, heads * vdim
    requests = Requests(gpu_device, (heads, dim, vdim), 4)
    want_state = [None] * 4
    gen = torch.Generator().manual_seed(7)
    pad = 4 if dim % 4 == 0 else 3                         # rows that can be read 16 bytes wide, or not
    pairs = dim // 2 - (dim // 2 > 3)
    angles = torch.outer(torch.arange(400.0), 0.3 ** torch.arange(pairs))
    table = torch.stack([angles.cos(), angles.sin()], -1).contiguous()
    for spans in SPANS:
        batch = requests.step(spans)
        T = batch.num_tokens
        x = torch.randn(T, pad + 2 * qk + inner, generator=gen)
        kw = dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, silu_inputs=mode == "fixed")
        if mode == "turned" and pairs > 0:
            kw.update(turn=table.to(gpu_device), k_scale=0.5)
        beta = None
        if mode in ("fixed", "turned"):
            decay = torch.tensor([1.0, 0.0, 0.9, 0.999])[:heads]
            kw["decay"] = decay.to(gpu_device)
            g = decay.double()[None, :, None].expand(T, heads, 1)
        else:
            n = heads * dim if mode == "delta_per_channel" else heads
            gates = torch.cat([torch.rand(T, heads, generator=gen),
                               torch.rand(T, n, generator=gen) ** 0.1], 1)
            gates[T // 3, heads:] = 0.0                    # everything is forgotten
            gates[T // 2:, heads:] **= 20                  # and most of it in a few tokens
            kw.update(gates=gates.to(gpu_device), per_channel=n > heads,
                      delta=mode.startswith("delta"))
            g = gates[:, heads:].double().view(T, heads, -1)
            beta = gates[:, :heads].double() if kw["delta"] else None
        if beta is not None:                               # unit keys, as the rule has them
            k = x[:, pad + qk:pad + 2 * qk].view(T, kv_heads, dim)
            k /= k.norm(dim=-1, keepdim=True)
        xd = x.double()
        if mode == "fixed":
            xd = torch.nn.functional.silu(xd)
        q, k, v = xd[:, pad:pad + qk], xd[:, pad + qk:pad + 2 * qk], xd[:, pad + 2 * qk:]
        q, k = (t.reshape(T, kv_heads, dim).repeat_interleave(heads // kv_heads, 1) for t in (q, k))
        if "turn" in kw:
            pos = batch.positions.cpu().long()
            c, s = (table[pos, :, i].double()[:, None] for i in (0, 1))

            def turned(t):
                t = t.clone()
                even, odd = t[..., 0:2 * pairs:2].clone(), t[..., 1:2 * pairs:2].clone()
                t[..., 0:2 * pairs:2], t[..., 1:2 * pairs:2] = even * c - odd * s, odd * c + even * s
                return t
            q, k = turned(q), turned(k) * 0.5
        v = v.reshape(T, heads, vdim)
        x = x.to(gpu_device)
        (got, st), (walked, st_walked) = in_chunks_and_walked(
            ops, lambda: ops.linear_recurrence(x, pad, pad + qk, pad + 2 * qk, batch,
                                               requests.state, **kw), requests.state)
        at, want = 0, torch.empty(T, heads, vdim, dtype=torch.float64)
        for i, n in enumerate(spans):
            S = want_state[i] if want_state[i] is not None else torch.zeros(heads, dim, vdim,
                                                                            dtype=torch.float64)
            rows = slice(at, at + n)
            want[rows], want_state[i] = walk(q[rows], k[rows], v[rows], g[rows],
                                             None if beta is None else beta[rows], S)
            at += n
        no_further_off(got, walked, want.view(T, inner))
        slots = batch.slot_ids.long()
        no_further_off(st[slots], st_walked[slots], torch.stack(want_state))
        others = [i for i in range(st.shape[0]) if i not in slots.tolist()]
        assert (st[others] == 3.0).all()


@pytest.mark.parametrize("heads, groups, rows, vdim", [(8, 2, 128, 64), (3, 3, 10, 6), (4, 1, 200, 20),
                                                       (6, 1, 64, 33)])
def test_state_space_scan_in_chunks(gpu_device, heads, groups, rows, vdim):
    ops = load_hip_ops(gpu_device)
    inner, gen = heads * vdim, torch.Generator().manual_seed(8)
    requests = Requests(gpu_device, (heads, rows, vdim), 4)
    want_state = [torch.zeros(heads, rows, vdim, dtype=torch.float64) for _ in range(4)]
    bias, a_log, skip = (torch.randn(heads, generator=gen) for _ in range(3))
    for spans in SPANS:
        batch = requests.step(spans)
        T = batch.num_tokens
        xbc = torch.randn(T, inner + 2 * groups * rows, generator=gen)
        proj = torch.randn(T, 5 + heads, generator=gen)
        args = [t.to(gpu_device) for t in (xbc, proj)]
        consts = [t.to(gpu_device) for t in (bias, a_log, skip)]
        (got, st), (walked, st_walked) = in_chunks_and_walked(
            ops, lambda: ops.ssm_scan(*args, 5, *consts, batch, requests.state, heads=heads,
                                      vdim=vdim, state_rows=rows, groups=groups), requests.state)
        d = torch.nn.functional.softplus(proj[:, 5:].double() + bias.double())
        g = torch.exp(-torch.exp(a_log.double()) * d)[..., None]
        x = xbc[:, :inner].double().view(T, heads, vdim)
        B, C = (t.reshape(T, groups, rows).repeat_interleave(heads // groups, 1)
                for t in xbc[:, inner:].double().split(groups * rows, 1))
        at, want = 0, torch.empty(T, heads, vdim, dtype=torch.float64)
        for i, n in enumerate(spans):
            r = slice(at, at + n)
            y, want_state[i] = walk(C[r], B[r], d[r][..., None] * x[r], g[r], None, want_state[i])
            want[r] = y + skip.double()[:, None] * x[r]
            at += n
        no_further_off(got, walked, want.view(T, inner))
        slots = batch.slot_ids.long()
        no_further_off(st[slots], st_walked[slots], torch.stack(want_state))


# (eight workgroups of 16 columns to every 64 tokens of the longest portion: two launches)
@pytest.mark.parametrize("mode, heads, kv_heads, dim, vdim", [
    ("per_head_plain", 32, 4, 20, 5), ("per_head_plain", 12, 3, 50, 40), ("per_head_plain", 8, 8, 128, 64),
    ("fixed", 4, 4, 20, 113), ("fixed", 4, 2, 50, 128), ("fixed", 4, 1, 100, 115),
    ("turned", 4, 4, 20, 128), ("turned", 4, 1, 65, 120), ("turned", 4, 2, 36, 113)])
def test_linear_recurrence_in_two_launches(gpu_device, mode, heads, kv_heads, dim, vdim):
    test_linear_recurrence_in_chunks(gpu_device, mode, heads, kv_heads, dim, vdim)


@pytest.mark.parametrize("heads, groups, rows, vdim", [(64, 8, 32, 16), (32, 4, 33, 15), (16, 2, 65, 18)])
def test_state_space_scan_in_two_launches(gpu_device, heads, groups, rows, vdim):
    test_state_space_scan_in_chunks(gpu_device, heads, groups, rows, vdim)


# (fewer than that at both of SPANS: three; heads that share q and k, 128 rows of S)
@pytest.mark.parametrize("mode", ["fixed", "per_head_plain", "turned"])
@pytest.mark.parametrize("vdim", [100, 128])
def test_linear_recurrence_in_three_launches(gpu_device, mode, vdim):
    test_linear_recurrence_in_chunks(gpu_device, mode, 2, 1, 128, vdim)


def test_state_space_scan_in_three_launches(gpu_device):
    test_state_space_scan_in_chunks(gpu_device, 4, 2, 128, 64)


def in_two_and_in_three(ops, monkeypatch, state, slot, batch, x, columns, **kw):
    """The output and the slot's state as a step makes them by itself, and beside a portion of 4,000 tokens
    (whose length says how many launches it is)."""
    scratch, make, before, results = [], ops._chunk_scratch, state.clone(), []
    # (scratch begins as a mark, so that what a form writes can be counted)
    monkeypatch.setitem(vars(ops), "_chunk_scratch",
                        lambda *args: scratch.append(make(*args).fill_(-2.0 ** 100)) or scratch[-1])
    monkeypatch.setattr(ops, "dispatch", dataclasses.replace(ops.dispatch, scan_whole_tokens=16))
    for longest in (batch.max_q_len, 4000):
        state.copy_(before)
        out = ops.linear_recurrence(x, *columns, dataclasses.replace(batch, max_q_len=longest, plans={}),
                                    state, silu_inputs=False, **kw)
        results.append((out, state[slot].clone()))
    two, three = ((s != -2.0 ** 100).sum().item() for s in scratch)
    assert two != three
    return results


@pytest.mark.parametrize("heads, kv_heads, dim, vdim", [(8, 2, 128, 128), (12, 4, 40, 50), (8, 8, 64, 80)])
@pytest.mark.parametrize("tokens", [40, 200, 300])
def test_two_launches_and_three_give_the_same_bits(gpu_device, monkeypatch, tokens, heads, kv_heads, dim, vdim):
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(17)
    requests = Requests(gpu_device, (heads, dim, vdim), 1)
    x = torch.randn(2, tokens, 2 * kv_heads * dim + heads * vdim, generator=gen).to(gpu_device)
    gates = torch.cat([torch.rand(tokens, heads, generator=gen),
                       torch.rand(tokens, heads, generator=gen) ** 0.1], 1).to(gpu_device)
    for rows in x:                                         # at position 0, and behind that
        batch = requests.step([tokens])
        two, three = in_two_and_in_three(
            ops, monkeypatch, requests.state, batch.slot_ids[0].item(), batch, rows,
            (0, kv_heads * dim, 2 * kv_heads * dim), heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim,
            gates=gates)
        assert torch.equal(two[0], three[0]) and torch.equal(two[1], three[1])
        monkeypatch.undo()


# 2^24 times four decays whose product in 64 bits, then rounded to 32, hangs on the order (for all tokens
# but four the decay is 1)
ROUNDED_APART = {
    "tokens 1 to 4": [(8455556, 16707183, 16586236, 11763250), (14533896, 15783492, 11605631, 12895099)],
    "a block each": [(10746809, 12595570, 9500064, 14306753), (11433115, 11517348, 10958803, 13946748),
                     (14191418, 13858469, 13507899, 10767477), (13046945, 8467980, 9204622, 11222547)]}


def test_two_launches_and_three_multiply_decays_in_one_order(gpu_device, monkeypatch):
    """Every k and q a unit vector and v of one token alone: outputs and state are that token's decays."""
    ops = load_hip_ops(gpu_device)
    heads, dim, vdim, tokens = 16, 16, 16, 128
    gates, v = torch.ones(tokens, 2 * heads), torch.zeros(tokens, heads, vdim)
    planted = [(place, four, chunk) for place, fours in ROUNDED_APART.items() for four in fours
               for chunk in (0, 64)]
    v[0] = 1
    for h, (place, four, chunk) in enumerate(planted):     # in the chunk of that v, or in the one behind it
        at = (1, 2, 3, 4) if place == "tokens 1 to 4" else (5, 20, 40, 50)
        gates[[chunk + t for t in at], heads + h] = torch.tensor(four) / 2.0 ** 24
    x = torch.cat([torch.eye(1, dim).expand(tokens, dim)] * 2 + [v.view(tokens, -1)], 1).contiguous()
    requests = Requests(gpu_device, (heads, dim, vdim), 1)
    batch = requests.step([tokens])
    two, three = in_two_and_in_three(
        ops, monkeypatch, requests.state, batch.slot_ids[0].item(), batch, x.to(gpu_device), (0, dim, 2 * dim),
        heads=heads, kv_heads=1, dim=dim, vdim=vdim, gates=gates.to(gpu_device))
    assert torch.equal(two[0], three[0]) and torch.equal(two[1], three[1])
    # and to 32 bits what 64 give: two to four products rounded to 53, one to 24
    want = torch.cumprod(gates[:, heads:].double(), 0)
    got = two[0].double().cpu().view(tokens, heads, vdim)[:, :, 0]
    assert ((got - want).abs() <= 2.0 ** -22 * want).all()


@pytest.mark.parametrize("tokens", [16, 17, 63, 64, 65, 128, 129, 192, 193, 209, 272])
def test_two_launches_at_every_number_of_chunks(gpu_device, tokens):
    """The walk's loops turn by turn: one chunk to five, the last of one tile, of more, whole."""
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(15)
    heads, dim, vdim = 40, 40, 17
    requests = Requests(gpu_device, (heads, dim, vdim), 2)
    spans = [tokens, 1]
    batch = requests.step(spans)
    x = torch.randn(sum(spans), heads * (2 * dim + vdim), generator=gen)
    gates = torch.cat([torch.rand(sum(spans), heads, generator=gen),
                       torch.rand(sum(spans), heads, generator=gen) ** 0.1], 1)
    x_dev, gates_dev = x.to(gpu_device), gates.to(gpu_device)
    (got, st), (walked, st_walked) = in_chunks_and_walked(
        ops, lambda: ops.linear_recurrence(
            x_dev, 0, heads * dim, 2 * heads * dim, batch, requests.state, heads=heads, kv_heads=heads,
            dim=dim, vdim=vdim, silu_inputs=False, gates=gates_dev), requests.state)
    q, k, v = x.double().split([heads * dim] * 2 + [heads * vdim], 1)
    q, k, v = q.view(-1, heads, dim), k.view(-1, heads, dim), v.view(-1, heads, vdim)
    g, at, want, states = gates[:, heads:, None].double(), 0, [], []
    for n in spans:
        r = slice(at, at + n)
        out, S = walk(q[r], k[r], v[r], g[r], None, torch.zeros(heads, dim, vdim, dtype=torch.float64))
        want.append(out)
        states.append(S)
        at += n
    no_further_off(got, walked, torch.cat(want).view(at, -1))
    slots = batch.slot_ids.long()
    no_further_off(st[slots], st_walked[slots], torch.stack(states))


@pytest.mark.parametrize("what", ["q", "k", "v"])
def test_two_launches_keep_what_is_not_finite_from_earlier_tokens(gpu_device, what):
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(16)
    kept, spans = ops.dispatch, [150, 70]
    heads, kv_heads, dim, vdim = 16, 4, 64, 33
    x = torch.randn(sum(spans), 2 * kv_heads * dim + heads * vdim, generator=gen)
    decay = 0.9 + 0.02 * torch.randn(heads, generator=gen).tanh().to(gpu_device)
    column = {"q": 0, "k": kv_heads * dim, "v": 2 * kv_heads * dim}[what]

    def run(x):
        requests = Requests(gpu_device, (heads, dim, vdim), 2)
        batch = requests.step(spans)
        ops.dispatch = dataclasses.replace(kept, scan_whole_tokens=16)
        try:
            return ops.linear_recurrence(
                x.to(gpu_device), 0, kv_heads * dim, 2 * kv_heads * dim, batch, requests.state,
                heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, silu_inputs=False, decay=decay)
        finally:
            ops.dispatch = kept

    want = run(x)
    for t in (0, 5, 37, 63, 64, 79, 140):
        for value in (float("inf"), float("nan")):
            xs = x.clone()
            xs[t, column] = value
            out = run(xs)
            assert torch.equal(out[:t], want[:t]) and torch.equal(out[150:], want[150:]), (t, value)
            assert not out[t].isfinite().all(), (t, value)
            if what == "q":
                assert torch.equal(out[t + 1:], want[t + 1:]), (t, value)


@pytest.mark.parametrize("per_channel", [False, True])
def test_delta_rule_takes_silu_of_its_operands_in_long_portions(gpu_device, per_channel):
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(9)
    heads, dim, vdim = 2, 36, 20
    requests, spans = Requests(gpu_device, (heads, dim, vdim), 2), [150, 70]
    batch = requests.step(spans)
    T, n = batch.num_tokens, heads * dim if per_channel else heads
    x = torch.randn(T, heads * (2 * dim + vdim), generator=gen)
    x[:, :2 * heads * dim] *= 0.2
    gates = torch.cat([torch.rand(T, heads, generator=gen), torch.rand(T, n, generator=gen) ** 0.1], 1)
    out = ops.linear_recurrence(
        x.to(gpu_device), 0, heads * dim, 2 * heads * dim, batch, requests.state, heads=heads,
        kv_heads=heads, dim=dim, vdim=vdim, silu_inputs=True, delta=True, per_channel=per_channel,
        gates=gates.to(gpu_device))
    q, k, v = torch.nn.functional.silu(x.double()).split([heads * dim] * 2 + [heads * vdim], 1)
    q, k, v = q.view(T, heads, dim), k.view(T, heads, dim), v.view(T, heads, vdim)
    g, beta = gates[:, heads:].double().view(T, heads, -1), gates[:, :heads].double()
    want, at = [], 0
    for rows in spans:
        r = slice(at, at + rows)
        want.append(walk(q[r], k[r], v[r], g[r], beta[r],
                         torch.zeros(heads, dim, vdim, dtype=torch.float64))[0])
        at += rows
    torch.testing.assert_close(out.double().cpu(), torch.cat(want).view(T, -1), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("tokens", [3, 200])
def test_states_of_more_rows_are_refused_with_a_message(gpu_device, tokens):
    ops = load_hip_ops(gpu_device)
    heads, rows, vdim = 2, 260, 4
    requests = Requests(gpu_device, (heads, rows, vdim), 1)
    batch = requests.step([tokens])
    xbc = torch.zeros(tokens, heads * vdim + 2 * rows, device=gpu_device)
    proj, consts = torch.zeros(tokens, heads, device=gpu_device), torch.zeros(heads, device=gpu_device)
    with pytest.raises(KernelError, match="260"):
        ops.ssm_scan(xbc, proj, 0, consts, consts, consts, batch, requests.state, heads=heads,
                     vdim=vdim, state_rows=rows, groups=1)


@pytest.mark.parametrize("what", ["q", "k", "v", "gates"])
@pytest.mark.parametrize("mode", ["fixed", "turned", "per_head", "delta", "delta_per_channel", "scan"])
def test_what_is_not_finite_does_not_reach_earlier_tokens(gpu_device, mode, what):
    """Infinities and NaN in a token's operands: the tokens before it and the other requests come
    out the same to the bit, a q reaches its own token alone."""
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(10)
    ops_dispatch = dataclasses.replace(ops.dispatch, scan_whole_tokens=16, state_space_whole_tokens=16)
    heads, kv_heads, dim, vdim, spans = 4, 2, 64, 33, [150, 70]
    n_gates = heads * dim if mode == "delta_per_channel" else heads
    x = torch.randn(sum(spans), 2 * kv_heads * dim + heads * vdim, generator=gen)
    x[:, :2 * kv_heads * dim] *= 0.15
    gates = torch.cat([torch.rand(sum(spans), heads, generator=gen),
                       torch.rand(sum(spans), n_gates, generator=gen) ** 0.1], 1)
    q_col, k_col, v_col = 0, kv_heads * dim, 2 * kv_heads * dim
    if mode == "scan":                                     # x | B | C, and the step sizes
        v_col, k_col, q_col = 0, heads * vdim, heads * vdim + kv_heads * dim
    column = {"q": q_col, "k": k_col, "v": v_col}
    consts = [torch.randn(heads, generator=gen).to(gpu_device) for _ in range(3)]
    angles = torch.outer(torch.arange(200.0), 0.3 ** torch.arange(dim // 2))
    table = torch.stack([angles.cos(), angles.sin()], -1).contiguous().to(gpu_device)

    def run(x, gates):
        requests = Requests(gpu_device, (heads, dim, vdim), 2)
        batch, kept = requests.step(spans), ops.dispatch
        x, gates = x.to(gpu_device), gates.to(gpu_device)
        ops.dispatch = ops_dispatch
        try:
            if mode == "scan":
                return ops.ssm_scan(x, gates, heads, *consts, batch, requests.state, heads=heads,
                                    vdim=vdim, state_rows=dim, groups=kv_heads)
            kw = dict(gates=gates, per_channel=n_gates > heads, delta=mode.startswith("delta"))
            if mode in ("fixed", "turned"):
                kw = dict(decay=0.9 + 0.02 * consts[0].tanh(), silu_inputs=mode == "fixed")
            if mode == "turned":
                kw.update(turn=table, k_scale=0.5)
            return ops.linear_recurrence(x, q_col, k_col, v_col, batch, requests.state, heads=heads,
                                         kv_heads=kv_heads, dim=dim, vdim=vdim,
                                         **{"silu_inputs": False, **kw})
        finally:
            ops.dispatch = kept

    want = run(x, gates)
    for t in (0, 5, 37, 63, 64, 79, 140):
        for value in (float("inf"), float("nan")):
            xs, gs = x.clone(), gates.clone()
            if what == "gates":
                if mode in ("fixed", "turned"):
                    return
                gs[t, heads:] = value
            else:
                xs[t, column[what]] = value
            out = run(xs, gs)
            assert torch.equal(out[:t], want[:t]), (t, value)
            assert torch.equal(out[150:], want[150:]), (t, value)
            assert not out[t].isfinite().all() or (mode == "scan" and what == "gates"), (t, value)
            if what == "q":
                assert torch.equal(out[t + 1:], want[t + 1:]), (t, value)


@pytest.mark.parametrize("shift", [6, 9, 11])
def test_equal_decays_do_not_add_up_their_roundings(gpu_device, shift):
    """A chunk's whole decay is rounded once, by 2^-24 of itself at most, and what is j chunks old
    has met it j times: 1 / (1 - g^64) times on average; beside it the sums' own roundings (the mean
    square of 64 in a chain is 32, each less than 0.45 x 2^-24; as many again for the products)."""
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(11)
    heads, dim, vdim, T, g = 2, 64, 32, 1500, 1 - 2.0 ** -shift
    requests = Requests(gpu_device, (heads, dim, vdim), 1)
    batch = requests.step([T])
    x = torch.randn(T, heads * (2 * dim + vdim), generator=gen)
    x[:, :2 * heads * dim] *= dim ** -0.25
    out = ops.linear_recurrence(
        x.to(gpu_device), 0, heads * dim, 2 * heads * dim, batch, requests.state, heads=heads,
        kv_heads=heads, dim=dim, vdim=vdim, silu_inputs=False,
        decay=torch.full((heads,), g).to(gpu_device))
    q, k, v = x.double().split([heads * dim] * 2 + [heads * vdim], 1)
    want, S = walk(q.view(T, heads, dim), k.view(T, heads, dim), v.view(T, heads, vdim),
                   torch.full((T, heads, 1), g, dtype=torch.float64), None,
                   torch.zeros(heads, dim, vdim, dtype=torch.float64))
    bound = 2.0 ** -24 * (1 / (1 - g ** 64) + 0.45 * 64 ** 0.5)
    state = requests.state[batch.slot_ids.long()][0].double().cpu()
    assert (state - S).norm() <= bound * S.norm()
    want = want.view(T, -1)
    assert (out.double().cpu() - want).norm() <= 2 * bound * want.norm()


@pytest.mark.parametrize("mode", ["per_head", "delta", "delta_per_channel"])
def test_chunks_round_no_more_than_the_walk_does(gpu_device, mode):
    """Additions of random signs, each off by less than 0.45 x 2^-24 of its sum in the mean square:
    128 products in chains of 8, their sums in pairs, give 4.5 + 1 + 4.5 such squares (q k, S q, W S
    in turn), 64 of them 4.5 + 1 + 2 (k u), and what a token reads has been through four such sums
    and some ten single roundings.  The outputs' error is the walk's to a few parts in a hundred
    (0.95 to 1.03 of it; 1.12 to 1.19 in chains of sixteen with decays multiplied up in 32 bits)."""
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(12)
    heads, dim, vdim, T = 2, 128, 64, 600
    n = heads * dim if mode == "delta_per_channel" else heads
    x = torch.randn(T, heads * (2 * dim + vdim), generator=gen)
    k = x[:, heads * dim:2 * heads * dim].view(T, heads, dim)
    k /= k.norm(dim=-1, keepdim=True)
    gates = torch.cat([torch.rand(T, heads, generator=gen), torch.rand(T, n, generator=gen) ** 0.05], 1)

    def run(walk):
        requests = Requests(gpu_device, (heads, dim, vdim), 1)
        batch = requests.step([T])
        out = ops.linear_recurrence(
            x.to(gpu_device), 0, heads * dim, 2 * heads * dim, batch, requests.state, heads=heads,
            kv_heads=heads, dim=dim, vdim=vdim, silu_inputs=False, delta=mode != "per_head",
            per_channel=n > heads, gates=gates.to(gpu_device), walk=walk)
        return out.double().cpu(), requests.state[batch.slot_ids.long()][0].double().cpu()

    q, k, v = x.double().split([heads * dim] * 2 + [heads * vdim], 1)
    want, S = walk(q.view(T, heads, dim), k.view(T, heads, dim), v.view(T, heads, vdim),
                   gates[:, heads:].double().view(T, heads, -1),
                   None if mode == "per_head" else gates[:, :heads].double(),
                   torch.zeros(heads, dim, vdim, dtype=torch.float64))
    bound = 0.45 * 2.0 ** -24 * (3 * 10 + 7.5 + 10) ** 0.5
    want = want.view(T, -1)
    (out, state), (walked, _) = run(False), run(True)
    off = (out - want).norm()
    assert off <= bound * want.norm()
    assert off <= 1.08 * (walked - want).norm()
    assert (state - S).norm() <= bound * S.norm()


@pytest.mark.parametrize("per_channel", [False, True])
def test_walked_portions_do_not_depend_on_the_cut(gpu_device, per_channel):
    """The same sums in the same order, so the same to the bit, for portions that the same number of
    lanes walks (from eight tokens on)."""
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(13)
    heads, dim, vdim, T = 3, 48, 40, 210
    n = heads * dim if per_channel else heads
    x = torch.randn(T, heads * (2 * dim + vdim), generator=gen)
    x[:, heads * dim:2 * heads * dim] *= dim ** -0.5
    gates = torch.cat([torch.rand(T, heads, generator=gen), torch.rand(T, n, generator=gen) ** 0.1], 1)
    x, gates = x.to(gpu_device), gates.to(gpu_device)

    def run(portions):
        requests, at, outs = Requests(gpu_device, (heads, dim, vdim), 1), 0, []
        for rows in portions:
            outs.append(ops.linear_recurrence(
                x[at:at + rows].contiguous(), 0, heads * dim, 2 * heads * dim, requests.step([rows]),
                requests.state, heads=heads, kv_heads=heads, dim=dim, vdim=vdim, silu_inputs=False,
                delta=True, per_channel=per_channel, gates=gates[at:at + rows].contiguous(), walk=True))
            at += rows
        assert at == T
        return torch.cat(outs)

    whole = run([T])
    for portions in ([70, 13, 127], [8, 9, 64, 129]):
        assert torch.equal(run(portions), whole), portions


@pytest.mark.parametrize("tokens, walked", [(128, True), (160, True), (161, False)])
def test_delta_rule_walks_portions_that_its_chunks_are_slower_for(gpu_device, tokens, walked):
    ops, gen = load_hip_ops(gpu_device), torch.Generator().manual_seed(14)
    heads, dim, vdim = 2, 64, 32
    x = torch.randn(tokens, heads * (2 * dim + vdim), generator=gen).to(gpu_device)
    x[:, heads * dim:2 * heads * dim] *= dim ** -0.5
    gates = torch.rand(tokens, 2 * heads, generator=gen).to(gpu_device)
    outs = []
    for walk in (False, True):
        requests = Requests(gpu_device, (heads, dim, vdim), 1)
        batch = requests.step([tokens])
        outs.append(ops.linear_recurrence(
            x, 0, heads * dim, 2 * heads * dim, batch, requests.state, heads=heads, kv_heads=heads,
            dim=dim, vdim=vdim, silu_inputs=False, delta=True, gates=gates, walk=walk))
        assert ("scan_chunks" in batch.plans) == (not walk and not walked)
    assert torch.equal(*outs) == walked
    torch.testing.assert_close(*outs, rtol=1e-4, atol=1e-4)
