"""The row-streaming kernels at rows that start at any element of a 128-byte line.

A row is streamed from its first 128-byte boundary in 16-byte chunks; the
elements before it and after the last whole chunk are read one by one.  Odd
vocabularies and offset views move every row's start; the sizes below are the
edges of that split and of the choice of workgroup size.

The oracle's float64 log-probs and entropies are compared at 2e-5 absolute:
the log-sum-exp is at most 16 in magnitude, where fp32 values are 1e-6 apart,
and the partial sums of up to 98305 terms add a relative error of a few 1e-7.
"""

import pytest
import torch

from oracle import logprob as olp

pytestmark = pytest.mark.gpu

TOL = 2e-5


def _logits(rows, T, V, offset, seed, dev):
    """[rows, T, V] bf16 logits that start `offset` elements into their storage,
    with each row's largest value among its first or last elements by turns."""
    g = torch.Generator().manual_seed(seed)
    flat = torch.randn(rows * T * V + offset, generator=g).mul_(2.0).to(torch.bfloat16)
    z = flat[offset:].view(rows, T, V)
    z[:, 0::2, 0] = 12.0
    z[:, 1::2, V - 1] = 12.0
    zd = flat.to(dev)[offset:].view(rows, T, V)
    return z, zd, torch.randint(0, V, (rows, T), generator=g)


@pytest.mark.parametrize("offset", [0, 1, 7, 8, 63])
@pytest.mark.parametrize("V", [1, 2, 63, 64, 65, 71, 127, 4099, 32832])
def test_forward_at_any_row_start(dev, V, offset):
    from meshy_amd import logprob

    z, zd, y = _logits(2, 5, V, offset, 100 * V + offset, dev)
    lp, ent = logprob.logprobs_and_entropy(zd, y.to(dev), with_entropy=True)
    ref = torch.log_softmax(z.double(), -1)
    assert (lp.cpu() - ref.gather(-1, y.unsqueeze(-1)).squeeze(-1)).abs().max().item() <= TOL
    assert (ent.cpu() + (ref.exp() * ref).sum(-1)).abs().max().item() <= TOL


# Both sides of the workgroup-size rule: up to 256 rows, more, and many rows of
# at least 3 full tiles.
@pytest.mark.parametrize("T,V", [(256, 4099), (257, 4099), (2047, 98305), (2048, 98303), (2048, 98305)])
def test_forward_on_both_sides_of_the_workgroup_size_rule(dev, T, V):
    from meshy_amd import logprob

    g = torch.Generator(device=dev).manual_seed(T + V)
    zd = torch.randn(1, T, V, generator=g, device=dev, dtype=torch.bfloat16).mul_(2.0)
    y = torch.randint(0, V, (1, T), generator=g, device=dev)
    lp, ent = logprob.logprobs_and_entropy(zd, y, with_entropy=True)
    rows = torch.cat([torch.arange(0, T, 97), torch.tensor([T - 1])])
    z, yr = zd[:, rows].cpu(), y[:, rows].cpu()
    assert (lp[:, rows].cpu() - olp.chunk_logprobs(z, yr, dtype=torch.float64)).abs().max().item() <= TOL
    assert (ent[:, rows].cpu() - olp.chunk_entropy(z, dtype=torch.float64)).abs().max().item() <= TOL
