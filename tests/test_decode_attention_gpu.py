"""The decode kernel where its work changes hands: every head size whose heads it norms and turns a few
lanes each, query rows up to and past what one turn of the preparing wavefront takes and up to and past
an element a thread of the merge, with key splits and without."""

import pytest
import torch

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
