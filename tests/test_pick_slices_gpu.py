"""The largest logit where a slice of the vocabulary begins and ends, on rows that do and do not
begin on 16 bytes: equal values by the lower index, infinities, what is not a number passed over."""

import pytest
import torch

from tokensprint_amd.kernels import load_hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("vocab", [1, 3, 255, 1028, 4095, 4096, 4097, 4100, 8192, 12289, 32000])
def test_argmax_at_the_edges_of_slices(gpu_device, vocab, offset):
    ops = load_hip_ops(gpu_device)
    rows = 9
    gen = torch.Generator().manual_seed(vocab)
    host = torch.randint(-40, 40, (rows, vocab), generator=gen).float()      # many equal values
    want = [int(torch.nonzero(row == row.max())[0]) for row in host]
    host[0], want[0] = -float("inf"), 0
    host[1, vocab - 1], want[1] = 99.0, vocab - 1
    host[2, vocab // 2], want[2] = float("inf"), vocab // 2
    if vocab > 1:
        host[3, 0] = float("nan")
        want[3] = 1 + int(torch.nonzero(host[3, 1:] == host[3, 1:].max())[0])
    flat = torch.empty(rows * vocab + offset, device=gpu_device)
    logits = flat[offset:].view(rows, vocab)
    logits.copy_(host)
    assert ops.argmax(logits).tolist() == want
    cold = torch.zeros(rows, device=gpu_device)
    keys = torch.arange(rows, device=gpu_device)
    assert ops.sample(logits, cold, keys).tolist() == want
