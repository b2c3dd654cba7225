"""Graph replays of GAE follow their inputs.

The scan's chunks meet in slots tagged with a number drawn per call, which a
captured launch carries into every replay; documents longer than a chunk make
every carry pass through a slot.  Each replay runs on other inputs than the one
before and must equal the eager call bit for bit (the carries are folded in a
fixed order).  From a replay with a non-finite value on, every replay takes the
exact pass that such a call is left to, whose order is another: at most 150
chunk maps composed as other trees of depth 16 and less, each rounding 2^-24 of
a partial sum that does not exceed the largest output by more than the rewards
and values it spans, here taken as twice.
"""
import pytest
import torch

from meshy_amd.gae import compute_returns, gae_and_returns

pytestmark = pytest.mark.gpu


def _fill(rewards, values, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    rewards.copy_((torch.rand(rewards.shape, generator=g, device=dev) < 0.05).float())
    values.copy_(torch.randn(values.shape, generator=g, device=dev))


def _same(got, want, exact, what):
    for a, b in zip(got, want):
        top = b[b.isfinite()].abs().max().item()
        torch.testing.assert_close(a, b, rtol=0, atol=0 if exact else 2 * 16 * 2.0 ** -24 * top, equal_nan=True,
                                   msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("rows,S,n_docs", [(1, 300_001, 3), (4, 65_536, 4), (1, 2048, 1)])
def test_replays_equal_eager_calls(dev, rows, S, n_docs):
    n = rows * S
    doc = (torch.arange(n, device=dev) * n_docs // n).view(rows, S)
    mask = torch.ones(rows, S, device=dev)
    rewards, values = torch.empty(2, rows, S, device=dev).unbind()
    _fill(rewards, values, 0, dev)

    def call():
        return *gae_and_returns(rewards, values, mask, doc, n_docs, gamma=0.999), compute_returns(rewards, mask, doc)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in range(1, 9):
        _fill(rewards, values, seed, dev)
        if seed == 5:
            values[0, S // 2] = float("nan")
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        _same(got, call(), seed < 5, f"replay {seed}")
        torch.cuda.synchronize()
