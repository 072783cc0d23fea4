"""The decode kernel where its work changes hands: every head size whose heads it norms and turns a few
lanes each, query rows up to and past what one turn of the preparing wavefront takes and up to and past
an element a thread of the merge, with key splits and without."""

import pytest
import torch

from scenarios import paged_scenario
from test_kernels_gpu import DECODE_SPANS, attend_decode_case
from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [32, 64, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 9, 16, 17])
def test_rows_and_head_sizes(gpu_device, hd, group):
    # one rounding to bfloat16 of the rotated heads, of the weights and of the result on both sides:
    # the bound that the decode form is held to at the other shapes
    ops = load_hip_ops(gpu_device)
    attend_decode_case(ops, gpu_device, torch.bfloat16, 2 * group, 2, hd, 16, None, DECODE_SPANS)
    # more items than the chip has units and at most 64 entries: ranked, no splits
    if group in (2, 17):
        attend_decode_case(ops, gpu_device, torch.bfloat16, 8 * group, 8, hd, 32, 300, DECODE_SPANS * 4)


@pytest.mark.parametrize("nq", [2, 4, 32])
@pytest.mark.parametrize("start", [0, 200])
def test_the_new_key_alone_in_reach(gpu_device, nq, start):
    """The step's own key has a finite score far below any stand-in for "no key", those before it lower
    ones still: its value, whichever way a workgroup's partial sums are merged (few rows, many)."""
    ops, nkv, hd = load_hip_ops(gpu_device), 2, 64
    batch, cache, table, _ = paged_scenario(gpu_device, torch.bfloat16, nkv=nkv, hd=hd, page_size=16,
                                            spans=[(start, 1)], seed=1)
    row = torch.randn(1, (nq + 2 * nkv) * hd, generator=torch.Generator().manual_seed(2)).bfloat16()
    row[:, :nq * hd], row[:, nq * hd:(nq + nkv) * hd] = 2.0 ** 60, -2.0 ** 50       # score -2^116
    cache.k_pages.fill_(-2.0 ** 60)                                                # -2^126
    got = ops.attend(row.to(gpu_device), batch, table, cache, True, num_heads=nq, num_kv_heads=nkv,
                     kv_in_row=nkv, head_dim=hd, q_weight=None, k_weight=None, eps=1e-6, cos_sin=None,
                     scale=1.0, window=None)
    value = row[:, (nq + nkv) * hd:].view(nkv, 1, hd).expand(-1, nq // nkv, -1).reshape(1, nq, hd)
    assert torch.equal(got.cpu(), value)
