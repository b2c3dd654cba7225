"""The masked document lengths that GAE counts from segment offsets.

The count reads groups of four positions with 16-byte loads, 8192 per step,
and what lies before and after them one by one, wherever the mask starts.
Documents start at every offset modulo 4 and have the lengths around those edges,
empty ones among them; with more than 2048 documents a wave takes one, and those
beyond 8192 tokens go to whole workgroups.  Counts of 0/1
masks are exact (lambda equals the fp32 formula of the exact count); sums of
fractional masks, up to 2^14 terms of at most 1 in fp32, lie within 2^-20
relative of float64, and lambda within that of 1 / (alpha L).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 4, 5, 0, 7, 2047, 2048, 2049, 0, 8191, 8192, 8193, 6, 16389, 3]


def _lambda(lengths, alpha=1.5, epsilon=1e-6):
    lam = 1.0 - 1.0 / (torch.tensor(alpha, dtype=lengths.dtype) * lengths.clamp(min=1))
    return lam.clamp(0.0, 1.0 - epsilon)


@pytest.mark.parametrize("lead", [0, 1, 2, 3])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("fractional", [False, True])
def test_lambda_of_counted_lengths(dev, lead, offset, fractional):
    from meshy_amd.gae import gae_and_returns

    g = torch.Generator().manual_seed(lead + 4 * offset)
    lengths = [lead] + LENGTHS
    n, total = len(lengths), sum(lengths)
    doc = torch.repeat_interleave(torch.arange(n), torch.tensor(lengths))
    flat = torch.rand(total + offset, generator=g)
    if not fractional:
        flat = (flat < 0.7).float()
    mask = flat.to(dev)[offset:].view(1, total)
    zeros = torch.zeros(1, total, device=dev)
    _, _, lam = gae_and_returns(zeros, zeros, mask, doc.view(1, -1).to(dev), n)
    counted = torch.zeros(n, dtype=torch.float64).index_add_(0, doc, flat[offset:].double())
    if fractional:
        err = (lam.cpu().double() - _lambda(counted)).abs()
        assert (err <= 2.0 ** -20 / counted.clamp(min=1) + 2.0 ** -23).all()
    else:
        assert torch.equal(lam.cpu(), _lambda(counted.float()))


@pytest.mark.parametrize("n", [2048, 2049, 2055, 9001])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_lambda_of_many_documents(dev, n, offset):
    from meshy_amd.gae import gae_and_returns

    g = torch.Generator().manual_seed(n + offset)
    lengths = torch.randint(0, 40, (n,), generator=g)
    lengths[[0, 7, n // 2, n - 1]] = torch.tensor([8192, 8193, 40000, 16411])  # a wave's last, and workgroups'
    total = int(lengths.sum())
    doc = torch.repeat_interleave(torch.arange(n), lengths)
    flat = (torch.rand(total + offset, generator=g) < 0.7).float()
    mask = flat.to(dev)[offset:].view(1, total)
    zeros = torch.zeros(1, total, device=dev)
    _, _, lam = gae_and_returns(zeros, zeros, mask, doc.view(1, -1).to(dev), n)
    counted = torch.zeros(n, dtype=torch.float64).index_add_(0, doc, flat[offset:].double())
    assert torch.equal(lam.cpu(), _lambda(counted.float()))
