"""The kernel of 32 query rows a wavefront that prompts' attention takes at head sizes 64 and 128:
each of its forms (one, two and four sets of wavefronts that split an item's keys) against the plain
attention, at the edges of its tiles (32 rows, items of 64 and 128), of its turns (32 and 64 keys) and
of pages, with every option that reaches it."""

import ctypes
import math
import time

import pytest
import torch

from kernel_refs import TorchOps
from scenarios import paged_scenario

pytestmark = pytest.mark.gpu

REF = TorchOps()
FORMS = {"one-set": 3, "two-sets": 4, "four-sets": 5}


@pytest.fixture(scope="module")
def ops(gpu_device):
    from tokensprint_amd.kernels import load_hip_ops
    return load_hip_ops(gpu_device)


@pytest.fixture(params=FORMS.values(), ids=FORMS.keys())
def form(ops, request):
    ops.lib.ts_attention_prefill_variant(request.param)
    yield request.param
    ops.lib.ts_attention_prefill_variant(2)


def rand(shape, device, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(device)


def check(ops, device, nq, nkv, hd, page, spans, **options):
    """bfloat16 outputs against float32 attention over the same bfloat16 operands: weights are
    rounded to 8 bits (2^-9 of the largest value each, at random) and so is the result (2^-9)."""
    batch, cache, table, _ = paged_scenario(device, torch.bfloat16, nkv=nkv, hd=hd, page_size=page,
                                            spans=spans, seed=11)
    assert ops._prefill_tiles(batch, nkv, nq // nkv) is not None
    q = rand((batch.num_tokens, nq, hd), device, 12).bfloat16()
    kw = dict(num_heads=nq, num_kv_heads=nkv, head_dim=hd, scale=hd ** -0.5, window=None)
    kw.update(options)
    got = ops.paged_attention(q, batch, table, cache, **kw)
    T, only, first = batch.num_tokens, set(), 0
    for _, n in spans:          # a span's ends and the tokens around borders of items and tiles
        only |= {first + t for t in (0, 1, 7, 8, 15, 16, 31, 32, 63, 64, 127, 128, n // 2, n - 2, n - 1)
                 if 0 <= t < n}
        first += n
    only = sorted(only)
    want = REF.paged_attention(q, batch, table, cache, only=only, **kw)
    torch.testing.assert_close(got[only].float(), want[only].float(), rtol=1.6e-2, atol=1.6e-2)
    assert torch.isfinite(got.float()).all()
    return got, T


@pytest.mark.parametrize("nq,nkv,hd,page", [(16, 8, 128, 16), (8, 8, 64, 16), (24, 8, 128, 32),
                                            (32, 4, 64, 64), (40, 2, 128, 16), (16, 1, 128, 128)])
@pytest.mark.parametrize("spans", [
    [(0, 1000), (333, 1), (64, 33), (31, 65), (0, 17)],
    [(448, 515), (63, 64), (1023, 1), (17, 191)],
], ids=["from-the-start", "behind-others"])
def test_spans(ops, gpu_device, form, nq, nkv, hd, page, spans):
    check(ops, gpu_device, nq, nkv, hd, page, spans)


@pytest.mark.parametrize("options", [
    dict(window=1), dict(window=33), dict(window=200), dict(chunk=96), dict(window=40, keep_first=5),
    dict(window=100, keep_first=70), dict(chunk=64, keep_first=130), dict(scale=2.5), dict(softcap=3.0),
    dict(q_temp=(0.3, 100)), dict(softcap=20.0, window=90, keep_first=3),
], ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()))
@pytest.mark.parametrize("nq,nkv,hd", [(16, 8, 128), (12, 4, 64)])
def test_options(ops, gpu_device, form, nq, nkv, hd, options):
    check(ops, gpu_device, nq, nkv, hd, 16, [(0, 700), (450, 1), (300, 260)], **options)


@pytest.mark.parametrize("hd", [64, 128])
def test_sinks_and_slopes(ops, gpu_device, form, hd):
    sink, slopes = rand((16,), gpu_device, 13, 2.0), rand((16,), gpu_device, 14).abs() * 0.05
    check(ops, gpu_device, 16, 8, hd, 16, [(0, 600), (100, 200)], sink=sink)
    check(ops, gpu_device, 16, 8, hd, 16, [(0, 600), (100, 200)], slopes=slopes, sink=sink)


def test_growing_scores(ops, gpu_device, form):
    """Scores that rise along the keys, by far more than a weight's range, and fall again: every block
    brings new largest scores for some rows, or none."""
    nq, nkv, hd, S = 16, 8, 128, 900
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=nkv, hd=hd, page_size=16,
                                            spans=[(0, S)], seed=15)
    direction = rand((hd,), gpu_device, 16)
    direction = direction / direction.norm()
    q = (rand((S, nq, hd), gpu_device, 17) * 0.3 + 4.0 * direction).bfloat16()
    for shape in (lambda x: x, lambda x: 1 - x, lambda x: (x * 6).sin()):
        for page in range(-(-S // 16)):
            x = (torch.arange(16, device=gpu_device) + page * 16) / S
            k = rand((nkv, 16, hd), gpu_device, 18 + page) * 0.2 + shape(x)[:, None] * 12.0 * direction
            cache.k_pages[table[0, page]] = k.bfloat16()
        kw = dict(num_heads=nq, num_kv_heads=nkv, head_dim=hd, scale=1.0, window=None)
        got = ops.paged_attention(q, batch, table, cache, **kw)
        only = list(range(0, S, 13)) + [31, 32, 63, 64, S - 1]
        want = REF.paged_attention(q, batch, table, cache, only=only, **kw)
        # (a few keys hold most of the weight, so the weights' rounding does not average out: 2^-8 of
        # values up to 4)
        torch.testing.assert_close(got[only].float(), want[only].float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("sharpness", [1.0, 3.0, 8.0])
@pytest.mark.parametrize("hd", [64, 128])
def test_error_against_float64(ops, gpu_device, form, hd, sharpness):
    """How far outputs are from float64: the rounding of the result and of the weights, but not of a row's
    largest weight, which is one.  A relative rounding to 8 bits has a root mean square of
    2^-7 / sqrt(12) sqrt(E[1 / m^2]), m spread over [1, 2) as a logarithm's: 1.66e-3; errors of different weights
    add as squares.  (With the largest weight rounded too, rows that few keys dominate are 1.14 to 1.25 times as far.)"""
    nq, nkv, start, n = 16, 8, 512, 700
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=nkv, hd=hd, page_size=16,
                                            spans=[(start, n)], seed=21)
    q = rand((n, nq, hd), gpu_device, 22, sharpness).bfloat16()
    got = ops.paged_attention(q, batch, table, cache, num_heads=nq, num_kv_heads=nkv, head_dim=hd,
                              scale=hd ** -0.5, window=None)
    pages = table[0, :-(-(start + n) // 16)].long()
    k = cache.k_pages[pages].double().permute(1, 0, 2, 3).reshape(nkv, -1, hd)[:, :start + n]
    v = cache.v_pages[pages].double().permute(1, 0, 3, 2).reshape(nkv, -1, hd)[:, :start + n]
    hidden = (torch.arange(start + n, device=gpu_device)[None, :]
              > (start + torch.arange(n, device=gpu_device))[:, None])
    off = size = weights = 0.0
    for h in range(nq):
        scores = q[:, h].double() @ k[h // 2].T.contiguous() * hd ** -0.5
        w = scores.masked_fill(hidden, float("-inf")).softmax(-1)
        want = w @ v[h // 2]
        off += (got[:, h].double() - want).square().sum().item()
        size += want.square().sum().item()
        w.scatter_(1, w.argmax(1, keepdim=True), 0.0)
        weights += (w.square() @ v[h // 2].square()).sum().item()
    rounding = 2.0 ** -7 / 12 ** 0.5 * (0.375 / math.log(2)) ** 0.5
    assert off ** 0.5 <= 1.05 * rounding * (size + weights) ** 0.5


def test_the_same_every_time(ops, gpu_device, form):
    """Waves with blocks to skip run ahead of the others of their workgroup; a block sent for too
    early would show as a result that differs from launch to launch."""
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=8, hd=128, page_size=16,
                                            spans=[(0, 1212), (333, 1), (50, 1027)], seed=19)
    q = rand((batch.num_tokens, 16, 128), gpu_device, 20).bfloat16()
    for window in (None, 40, 333):
        kw = dict(num_heads=16, num_kv_heads=8, head_dim=128, scale=128 ** -0.5, window=window)
        first = ops.paged_attention(q, batch, table, cache, **kw).clone()
        for _ in range(20):
            assert torch.equal(ops.paged_attention(q, batch, table, cache, **kw), first)


def test_which_form(ops):
    """The plan of a step: sets by how many items there are and how long they are."""
    def plan(q_lens, starts, head_dim=128, page=16, heads=8, reach=0, rows=2):
        n, sets = len(q_lens), ctypes.c_int(-1)
        tiles = ops.lib.ts_attention_prefill_plan(head_dim, page, rows, heads, reach, n,
                                                  (ctypes.c_int * n)(*q_lens), (ctypes.c_int * n)(*starts),
                                                  ctypes.byref(sets))
        return tiles, sets.value
    assert plan([1024], [0]) == (4, 4)
    assert plan([2600], [0]) == (8, 2)
    assert plan([8192], [0], rows=8) == (8, 1)
    # under a window the items are short, however long the sequence: one round is not what decides
    assert plan([8192], [0], reach=128) == (8, 1)
    assert plan([1] * 200, [4000] * 200) == (4, 0)
    assert plan([1024], [0], head_dim=96) == (4, 0)
    assert plan([1024], [0], page=24) == (1, 0)


def plan_of(ops, q_lens, starts, head_dim=128, heads=8, rows=2, scores=False):
    n, sets = len(q_lens), ctypes.c_int(-1)
    choose = ops.lib.ts_attention_prefill_plan_scores if scores else ops.lib.ts_attention_prefill_plan
    tiles = choose(head_dim, 16, rows, heads, 0, n, (ctypes.c_int * n)(*q_lens), (ctypes.c_int * n)(*starts),
                   ctypes.byref(sets))
    return tiles, sets.value


@pytest.mark.parametrize("lanes, ctx, portion", [(200, 300, 33), (400, 300, 33), (200, 300, 256), (400, 1500, 33)])
def test_single_tokens_are_most_of_the_work(ops, lanes, ctx, portion):
    """A portion beside many single tokens does not take their kernel from them; it does where it is most
    of the work, or where scores are more than a product and that kernel is the slower one."""
    for head_dim in (64, 128):
        q_lens, starts = [1] * lanes + [portion], [ctx] * lanes + [0]
        assert plan_of(ops, q_lens, starts, head_dim) == (4, 0)
        assert plan_of(ops, [1] * 12 + [2000], [ctx] * 12 + [0], head_dim)[1] > 0
    assert plan_of(ops, q_lens, starts, 128, scores=True)[1] > 0
    if ctx == 300:
        assert plan_of(ops, q_lens, starts, 64, scores=True) == (4, 0)


def test_what_a_plan_costs(ops):
    """Many items for many units (one key/value head): each goes to the unit that is free first out of a
    heap, where a look at all units for every item took 0.8 to 1.2 ms."""
    for q_lens, starts in (([1] * 1000 + [33], list(range(1000)) + [0]), ([8192], [0])):
        least = float("inf")
        for _ in range(20):
            t = time.perf_counter()
            plan_of(ops, q_lens, starts, heads=1, rows=16)
            least = min(least, time.perf_counter() - t)
        assert least < 5e-4


@pytest.mark.parametrize("nq, nkv, hd", [(16, 8, 64), (16, 8, 128), (24, 3, 64)])
@pytest.mark.parametrize("options", [{}, dict(window=40, keep_first=5), dict(softcap=3.0)], ids=str)
def test_many_single_tokens_beside_a_portion(ops, gpu_device, nq, nkv, hd, options):
    spans = [((37 * i) % 600, 1) for i in range(210)] + [(130, 45), (0, 33)]
    if not options:
        rows = nq // nkv
        assert plan_of(ops, [n for _, n in spans], [s for s, _ in spans], hd, nkv, rows) == (4, 0) or nkv == 3
    check(ops, gpu_device, nq, nkv, hd, 16, spans, **options)
