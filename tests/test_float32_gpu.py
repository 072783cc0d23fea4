"""The float32 path's products and attention on the float32 matrix cores, at the edges of their
tiles, runs of K and key blocks: against float64, and a row the same to the bit however it is
batched."""

import ctypes

import pytest
import torch

from scenarios import paged_scenario
from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu

#: tiles of the product cut in parts; the first ones take 16, 32, ... rows at most
TILES, ROW_TILES = 10, 3


def rand(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("K", [4, 12, 16, 20, 124, 128, 132, 512, 1024, 1092, 3072])
@pytest.mark.parametrize("N", [5, 64, 150, 4100])
def test_product_rows_do_not_depend_on_the_number_of_rows(gpu_device, N, K):
    """Every kernel that a row count chooses (16, 32 and 64 rows, three tiles) and its edges."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((600, K), 1), rand((N, K), 2) * 0.05
    # |x| |w| summed, times a unit in the last place for every addition on an element's way
    bound = (x.abs().double() @ w.abs().double().T) * (2.0 ** -24) * (64 + 8 + K / 512)
    want = x.double() @ w.double().T
    x, w = x.to(gpu_device), w.to(gpu_device)
    full = ops.linear(x, w, torch.float32)
    assert ((full.double().cpu() - want).abs() <= bound).all()
    for M in (1, 8, 16, 17, 32, 33, 64, 65, 96, 129, 257):
        assert torch.equal(ops.linear(x[:M].contiguous(), w, torch.float32), full[:M]), M
        assert torch.equal(ops.linear(x[600 - M:].contiguous(), w, torch.float32), full[600 - M:]), M


@pytest.mark.parametrize("x_type, w_type", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("M", [3, 40, 70, 300])
def test_product_of_mixed_types(gpu_device, M, x_type, w_type):
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, 200), 3, x_type), (rand((150, 200), 4) * 0.05).to(w_type)
    want = x.double() @ w.double().T
    out = ops.linear(x.to(gpu_device), w.to(gpu_device), torch.float32)
    torch.testing.assert_close(out.double().cpu(), want, rtol=1e-5, atol=1e-5)


SPANS = [(0, 1), (63, 1), (64, 1), (0, 70), (15, 130), (500, 33), (0, 17)]


@pytest.mark.parametrize("nq, nkv, hd, page", [(16, 8, 128, 16), (6, 2, 48, 32), (5, 1, 16, 16),
                                               (4, 4, 64, 64), (16, 1, 80, 16), (7, 7, 112, 48)])
@pytest.mark.parametrize("form", ["plain", "window", "chunk_sink", "extras"])
def test_attention_against_the_general_kernel(gpu_device, monkeypatch, nq, nkv, hd, page, form):
    ops = load_hip_ops(gpu_device)
    batch, cache, table, _ = paged_scenario(gpu_device, torch.float32, nkv=nkv, hd=hd, page_size=page,
                                            spans=SPANS, seed=5)
    q = rand((batch.num_tokens, nq, hd), 6).to(gpu_device)
    kw = dict(num_heads=nq, num_kv_heads=nkv, head_dim=hd, scale=hd ** -0.5, window=None)
    if form == "window":
        kw["window"] = 37
    elif form == "chunk_sink":
        kw.update(chunk=50, sink=rand((nq,), 7).to(gpu_device))
    elif form == "extras":
        kw.update(softcap=3.0, slopes=(0.1 * rand((nq,), 8).abs()).to(gpu_device), q_temp=(0.3, 40),
                  window=200)
    assert ops.lib.ts_attention_f32_fits(hd, nq // nkv, page, nkv, 0) == 1
    # places behind an entry's last key hold whatever the page's last owner left
    for b, (start, n) in enumerate(SPANS):
        rest = (start + n) % page
        if rest:
            last = table[b, (start + n) // page].item()
            cache.k_pages[last, :, rest:] = float("nan")
            cache.v_pages[last, :, :, rest:] = float("nan")
    out = ops.paged_attention(q, batch, table, cache, **kw)
    monkeypatch.setattr(ops.lib, "ts_attention_f32_fits", lambda *a: 0)
    want = ops.paged_attention(q, batch, table, cache, **kw)
    torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-6)


def test_attention_of_a_token_does_not_depend_on_its_step(gpu_device):
    """Keys counted from position 0 in fixed blocks: a token alone, at the end of a portion and
    beside others adds up the same."""
    ops = load_hip_ops(gpu_device)
    kw = dict(num_heads=16, num_kv_heads=8, head_dim=128, scale=128 ** -0.5, window=None)
    batch, cache, table, _ = paged_scenario(gpu_device, torch.float32, nkv=8, hd=128, page_size=16,
                                            spans=[(0, 700), (40, 3)], seed=9)
    q = rand((batch.num_tokens, 16, 128), 10).to(gpu_device)
    for window in (None, 100):
        kw["window"] = window
        whole = ops.paged_attention(q, batch, table, cache, **kw)
        for t in (0, 63, 64, 333, 699):
            import copy
            one = copy.copy(batch)
            one.num_tokens = one.num_entries = one.max_q_len = 1
            one.q_lens, one.starts, one.plans = [1], [t], {}
            one.positions = batch.positions[t:t + 1].contiguous()
            one.entry_of_token = torch.zeros(1, dtype=torch.int32, device=gpu_device)
            one.q_start = torch.tensor([0, 1], dtype=torch.int32, device=gpu_device)
            one.ctx_len = torch.tensor([t + 1], dtype=torch.int32, device=gpu_device)
            alone = ops.paged_attention(q[t:t + 1].contiguous(), one, table[:1].contiguous(), cache, **kw)
            assert torch.equal(alone[0], whole[t]), t


@pytest.mark.parametrize("which", ["q", "k_pages", "v_pages"])
def test_attention_takes_buffers_that_do_not_begin_on_16_bytes(gpu_device, which):
    ops = load_hip_ops(gpu_device)
    kw = dict(num_heads=6, num_kv_heads=2, head_dim=32, scale=32 ** -0.5, window=None)
    batch, cache, table, _ = paged_scenario(gpu_device, torch.float32, nkv=2, hd=32, page_size=16,
                                            spans=[(0, 70), (33, 1), (5, 20)], seed=11)
    q = rand((batch.num_tokens, 6, 32), 12).to(gpu_device)
    want = ops.paged_attention(q, batch, table, cache, **kw)

    def moved(x):
        flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:]
        return flat.view(x.shape).copy_(x)

    if which == "q":
        q = moved(q)
    else:
        setattr(cache, which, moved(getattr(cache, which)))
    out = ops.paged_attention(q, batch, table, cache, **kw)
    torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-6)


@pytest.mark.parametrize("nq, nkv, hd, page", [(16, 8, 128, 16), (5, 1, 48, 32), (2, 2, 16, 16)])
@pytest.mark.parametrize("form", ["plain", "window", "chunk_sink"])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(gpu_device, monkeypatch, nq, nkv,
                                                                    hd, page, form):
    ops = load_hip_ops(gpu_device)
    spans = [(0, 130), (40, 37), (0, 9), (70, 1)]
    batch, cache, table, _ = paged_scenario(gpu_device, torch.float32, nkv=nkv, hd=hd, page_size=page,
                                            spans=spans, seed=13)
    q = rand((batch.num_tokens, nq, hd), 14).to(gpu_device)
    kw = dict(num_heads=nq, num_kv_heads=nkv, head_dim=hd, scale=hd ** -0.5, window=None)
    if form == "window":
        kw["window"] = 21
    elif form == "chunk_sink":
        kw.update(chunk=50, sink=rand((nq,), 15).to(gpu_device))
    finite = ops.paged_attention(q, batch, table, cache, **kw)
    spoilt = {0: [(45, float("inf")), (77, float("nan")), (101, float("-inf"))],
              1: [(60, float("nan"))], 2: [(5, float("inf"))], 3: [(3, float("inf"))]}
    for e, places in spoilt.items():
        for key, value in places:
            cache.v_pages[table[e, key // page].item(), -1, key % hd, key % page] = value
    cache.k_pages[table[0, 118 // page].item(), -1, 118 % page, 0] = float("nan")
    out = ops.paged_attention(q, batch, table, cache, **kw)
    monkeypatch.setattr(ops.lib, "ts_attention_f32_fits", lambda *a: 0)
    want = ops.paged_attention(q, batch, table, cache, **kw)
    torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-6, equal_nan=True)
    kept = out.isfinite()
    assert torch.equal(out[kept], finite[kept])
    assert kept[:45].all() and not kept.all()


@pytest.mark.parametrize("M", [1, 40, 501])
@pytest.mark.parametrize("N, K", [(1024, 1024), (512, 2048), (512, 3072)])
def test_product_rounds_no_more_than_short_chains_do(gpu_device, N, K, M):
    """Additions of random signs: a rounding is 2^-24 of what it rounds at most, in the mean square
    less than 0.45 of that, and K / 8 chains of eight products, a run's K / 128 steps and four
    pairs of runs give (8 / 2 + 1 + K / 256 + 3.5) such squares of the result's."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 16), rand((N, K), 17)
    want = x.double() @ w.double().T
    got = ops.linear(x.to(gpu_device), w.to(gpu_device), torch.float32).double().cpu()
    bound = 0.45 * 2.0 ** -24 * (8.5 + K / 256) ** 0.5 * 1.1
    assert (got - want).norm() <= bound * want.norm()


@pytest.mark.parametrize("K", [64, 192, 1088])
@pytest.mark.parametrize("M", [1, 17, 33, 64, 65, 200, 513])
@pytest.mark.parametrize("N", [3, 130, 1100])
def test_products_of_numbers_cut_in_three_parts(gpu_device, M, N, K):
    """Runs that are empty or shorter than others; results are not off to one
    side: the mean error of M N elements, each rounded by itself, is within five standard errors."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, K), 20).to(gpu_device), (rand((N, K), 21) * 0.05).to(gpu_device)
    want = x.double() @ w.double().T
    off = ops.linear(x, w, torch.float32).double() - want
    # a rounding of each of K / 32 sums in a run and of five sums of runs, three standard deviations
    # of a normal number times sqrt(K) 0.05, the largest of M N (less than 2^20) such
    assert float(off.abs().max()) <= 2.0 ** -24 * (K / 256 + 5) * 5.0 * K ** 0.5 * 0.05
    assert abs(float(off.mean())) <= 5.0 * float(off.pow(2).mean().sqrt()) / (M * N) ** 0.5 + 1e-12


@pytest.mark.parametrize("M", [9, 40, 70, 300])
def test_products_with_numbers_that_have_no_three_parts(gpu_device, M):
    """Infinities, NaN and numbers that bfloat16 rounds to an infinity: results as float32 has them."""
    ops = load_hip_ops(gpu_device)
    x, w = rand((M, 1024), 22), rand((300, 1024), 23)
    x[3, 5], x[4, 7], w[9, 100], x[6, 100], x[8, 2] = float("inf"), float("nan"), -3.4e38, 1.5, 3.402e38
    x[7], w[:, 2] = 0.0, 0.25
    want = (x.double() @ w.double().T).float()
    out = ops.linear(x.to(gpu_device), w.to(gpu_device), torch.float32).cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(torch.isinf(out), torch.isinf(want))
    fine = torch.isfinite(want)
    torch.testing.assert_close(out[fine], want[fine], rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("M", [1, 20, 40, 64, 70, 300, 600])
def test_a_row_of_a_single_product(gpu_device, M):
    """Nothing averages out: what is left out of a product of parts, 2^-25 of it twice at most, and
    one rounding, 2^-24, with a sixteenth of that for the roundings of the smaller parts."""
    ops = load_hip_ops(gpu_device)
    g = torch.Generator().manual_seed(24)
    x, w = torch.zeros(M, 1088), rand((1100, 1088), 25)
    x[torch.arange(M), torch.randint(0, 1088, (M,), generator=g)] = 1 + torch.rand(M, generator=g)
    w[7] = x[M - 1, x[M - 1].argmax()] = 1 + 2.0 ** -8 - 2.0 ** -23       # the parts behind the first are largest
    want = x.double() @ w.double().T
    got = ops.linear(x.to(gpu_device), w.to(gpu_device), torch.float32).double().cpu()
    assert ((got - want).abs() <= 2.1 * 2.0 ** -24 * want.abs()).all()


def by_tile(ops, x, w, tile, offset=0):
    """The product by a named tile, into a buffer that begins `offset` floats behind 16 bytes."""
    (M, K), N = x.shape, w.shape[0]
    out = torch.full((M * N + 8,), 7.0, device=x.device)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (x, w, out[offset:])]
    ops._call(ops.lib.ts_gemm_f32_split, *p, M, N, K, tile, ops._stream())
    assert (out[:offset] == 7).all() and (out[offset + M * N:] == 7).all()
    return out[offset:offset + M * N].view(M, N)


@pytest.mark.parametrize("tile", range(1, TILES + 1))
@pytest.mark.parametrize("K", [64, 192, 1088])
@pytest.mark.parametrize("N", [3, 130, 1100])
def test_every_tile_of_products_cut_in_parts(gpu_device, tile, N, K):
    """Each tile at its edges, with runs of K that are empty or shorter than others, equal to the bit
    to the largest one, whose sums are within a unit in the last place for every addition."""
    ops = load_hip_ops(gpu_device)
    for M in (1, 15, 16 * tile) if tile <= ROW_TILES else (1, 63, 133, 261):
        x, w = rand((M, K), 26).to(gpu_device), (rand((N, K), 27) * 0.05).to(gpu_device)
        whole = by_tile(ops, x, w, TILES)
        bound = (x.abs().double() @ w.abs().double().T) * 2.0 ** -24 * (10 + K / 256)
        assert ((whole.double() - x.double() @ w.double().T).abs() <= bound).all()
        assert torch.equal(by_tile(ops, x, w, tile), whole)
        assert torch.equal(by_tile(ops, x, w, tile, offset=1), whole)


@pytest.mark.parametrize("tile", range(1, TILES + 1))
@pytest.mark.parametrize("N", [203, 300])
def test_every_tile_with_numbers_that_have_no_three_parts(gpu_device, tile, N):
    ops = load_hip_ops(gpu_device)
    M = 16 * tile if tile <= ROW_TILES else 261
    x, w = rand((M, 192), 28), rand((N, 192), 29)
    x[3, 5], x[4, 7], w[9, 100], x[6, 100], x[8, 2] = float("inf"), float("nan"), -3.4e38, 1.5, 3.402e38
    x[7], w[:, 2], w[N - 1, 191], x[M - 1, 0] = 0.0, 0.25, float("nan"), float("-inf")
    want = (x.double() @ w.double().T).float()
    out = by_tile(ops, x.to(gpu_device), w.to(gpu_device), tile).cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(torch.isinf(out), torch.isinf(want))
    fine = torch.isfinite(want)
    torch.testing.assert_close(out[fine], want[fine], rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("tile", range(1, TILES + 1))
@pytest.mark.parametrize("K", [64, 1088])
def test_rows_and_columns_without_a_finite_result(gpu_device, tile, K):
    """Elements that are made again by a whole wavefront, all of a wavefront's and some of them,
    with fewer and with more fours of K than lanes."""
    ops = load_hip_ops(gpu_device)
    M, N = 16 * tile if tile <= ROW_TILES else 140, 133
    x, w = rand((M, K), 30), rand((N, K), 31)
    x[1], x[5, K - 1], w[16:40, 3], w[130, K - 4] = float("nan"), float("inf"), float("-inf"), float("nan")
    want = (x.double() @ w.double().T).float()
    out = by_tile(ops, x.to(gpu_device), w.to(gpu_device), tile).cpu()
    assert torch.equal(out.isnan(), want.isnan())
    fine = ~want.isnan()
    torch.testing.assert_close(out[fine], want[fine], rtol=1e-5, atol=1e-4)
