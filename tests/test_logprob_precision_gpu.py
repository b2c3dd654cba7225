"""The rounding error that the log-probs and the log-sum-exp keep.

Their last step carries the log-sum-exp in two fp32 parts, so that the result's
own rounding to fp32 (2^-24 relative at most, below 2^-25 in the 2-norm over many
values) and the sum's error (2^-24 of a sum s moves ln s by as much, small beside
values of magnitude 5 to 16) are what is left.  Rounded to one fp32 before the
difference is taken, a log-sum-exp adds an error of its own size: 3.1e-8 to 3.6e-8
here, against 2.5e-8 to 2.9e-8.
"""
import pytest
import torch

from meshy_amd import logprob, topk

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("n,V", [(64, 151936), (300, 151936), (2048, 131072), (1500, 50257), (8000, 100)])
def test_two_norm_error(dev, n, V):
    g = torch.Generator(device=dev).manual_seed(n + V)
    z = torch.randn(1, n, V, generator=g, device=dev).mul_(2.5).to(torch.bfloat16)
    ids = torch.randint(V, (1, n, 3), generator=g, device=dev)
    want = torch.empty(1, n, 3, dtype=torch.float64, device=dev)
    lse = torch.empty(1, n, dtype=torch.float64, device=dev)
    for i in range(0, n, 256):
        zd = z[:, i:i + 256].double()
        lse[:, i:i + 256] = torch.logsumexp(zd, -1)
        want[:, i:i + 256] = zd.gather(-1, ids[:, i:i + 256]) - lse[:, i:i + 256, None]
    assert _rel(logprob.logprobs_and_entropy(z, ids[..., 0]), want[..., 0]) <= 2.0 ** -25
    assert _rel(topk.gather_logprobs(z, ids), want) <= 2.0 ** -25
    assert _rel(logprob.logsumexp_rows(z), lse) <= 2.0 ** -25


# One logit above the others by 4 to 77: the sum's reference is the maximum of
# some elements, and an exponent d above it is rounded at 2^-24 d log2 e, so it
# may not lie far above: 2^-24 12 for the log-prob and, over the adds of a lane's
# and the waves' sums, a few times as much for the entropy, 2^-24 20 for the Top-K.
@pytest.mark.parametrize("n,V", [(37, 151936), (300, 50257), (2000, 50256), (2100, 131073), (5000, 100)])
def test_one_logit_above_the_others(dev, n, V):
    g = torch.Generator(device=dev).manual_seed(n)
    z = torch.randn(1, n, V, generator=g, device=dev).mul_(0.5).to(torch.bfloat16)
    y = torch.randint(V, (1, n), generator=g, device=dev)
    rows = torch.arange(0, n, max(1, n // 300), device=dev)
    for top in (4.0, 8.0, 10.0, 12.0, 14.0, 16.0, 20.125, 28.25, 40.0, 77.5):
        z.scatter_(-1, y[..., None], top)
        lp, ent = logprob.logprobs_and_entropy(z, y, with_entropy=True)
        best = topk.teacher_topk(z, 1)[1]
        ref = torch.log_softmax(z[:, rows].double(), -1)
        want = ref.gather(-1, y[:, rows, None])
        assert (lp <= 0).all(), top
        assert (lp[:, rows] - want[..., 0]).abs().max() <= 2.0 ** -20, top
        assert (best[:, rows] - want).abs().max() <= 2.0 ** -19, top
        assert (ent[:, rows] + (ref.exp() * ref).sum(-1)).abs().max() <= 2.0 ** -18, top
