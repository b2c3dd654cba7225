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


# Both sides of the bounds on rows, logits and ids that choose a workgroup's
# threads and loads for short and middle rows.
@pytest.mark.parametrize("T,V,K", [(257, 1024, 256), (257, 1025, 128), (257, 1025, 129), (257, 4097, 256), (4095, 8192, 9),
                                   (4096, 8192, 200), (4096, 8193, 9), (1024, 20001, 9), (1025, 20001, 9), (1025, 32767, 9), (1025, 32768, 9), (300, 36863, 9), (300, 36864, 9),
                                   (300, 98303, 9), (257, 131073, 200)])
def test_gather_on_both_sides_of_the_shape_rules(dev, T, V, K):
    from meshy_amd import logprob, topk

    g = torch.Generator(device=dev).manual_seed(T + V)
    zd = torch.randn(1, T, V + 1, generator=g, device=dev, dtype=torch.bfloat16).mul_(2.0)[..., 1:]
    ids = torch.randint(0, V, (1, T, K), generator=g, device=dev)
    out, lp = topk.gather_logprobs(zd, ids), logprob.logprobs_and_entropy(zd, ids[..., K - 1])
    rows = torch.cat([torch.arange(0, T, 97), torch.tensor([T - 1])]).to(dev)
    ref = torch.log_softmax(zd[:, rows].double(), -1).gather(-1, ids[:, rows])
    assert (out[:, rows] - ref).abs().max().item() <= TOL
    assert (lp[:, rows] - ref[..., K - 1]).abs().max().item() <= TOL


def _grad_ref(z, ids, g, lse):
    """float64 gradient of sum(g * (z[ids] - lse)) given the fp32 lse the kernel reads."""
    n, V = z.shape
    gd = torch.where(ids == -100, 0.0, g.double())
    out = -gd.sum(-1, keepdim=True) * (z.double() - lse.double().unsqueeze(-1)).exp()
    valid = (ids >= 0) & (ids < V)
    return out.scatter_add_(1, ids.clamp(0, V - 1), torch.where(valid, gd, 0.0))


def _check_backward(zd, ids, dev, seed):
    """Both backwards of [rows, T, V] logits at [rows, T, K] ids against float64:
    bf16 rounds to 2^-9 relative; the fp32 exponent of up to 16 and the sum of K
    gradients add less than 1e-5 of the largest gradient."""
    from meshy_amd import logprob, topk

    g = torch.Generator().manual_seed(seed)
    grad_out = torch.randn(ids.shape, generator=g)
    z = zd.detach().requires_grad_(True)
    out = topk.gather_logprobs(z, ids.to(dev))
    grads = [(torch.autograd.grad(out, z, grad_out.to(dev))[0], ids, grad_out)]
    lp = logprob.logprobs_and_entropy(z, ids[..., 0].to(dev))
    grads.append((torch.autograd.grad(lp, z, grad_out[..., 0].to(dev))[0], ids[..., :1], grad_out[..., :1]))
    lse = logprob.logsumexp_rows(zd).cpu()
    V = zd.shape[-1]
    for grad, i, go in grads:
        assert grad.is_contiguous() and grad.shape == zd.shape
        ref = _grad_ref(zd.cpu().reshape(-1, V), i.reshape(-1, i.shape[-1]), go.reshape(-1, i.shape[-1]), lse.reshape(-1))
        bad = ((i != -100) & ((i < 0) | (i >= V))).any(-1).reshape(-1)
        got = grad.cpu().reshape(-1, V).double()
        assert got[bad].isnan().all()
        err = (got - ref)[~bad].abs()
        assert (err <= 2.0 ** -8 * ref[~bad].abs() + 1e-5 * go.abs().max().item()).all()


def _ids(rows, T, K, V, seed):
    """Ids with duplicates, ignored ones, and at the row's first and last columns."""
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, V, (rows, T, K), generator=g)
    ids[:, 0, 0] = 0
    ids[:, -1, 0] = V - 1
    if K > 1:
        ids[:, 0, 1] = ids[:, 0, 0]
        ids[:, -1, K - 1] = -100
    if T > 2:
        ids[:, 1, 0] = -100
        ids[0, 2, K - 1] = V
    return ids


@pytest.mark.parametrize("K", [1, 9, 64, 65, 200])
@pytest.mark.parametrize("V", [1, 7, 255, 256, 257, 511, 519, 1001, 4099, 8192, 32003])
def test_backward_of_contiguous_logits(dev, V, K):
    # 3 * 7 * V elements: not a multiple of 8 for odd V, so the last chunk is partial.
    g = torch.Generator().manual_seed(V)
    zd = torch.randn(3, 7, V, generator=g).mul_(2.0).to(torch.bfloat16).to(dev)
    _check_backward(zd, _ids(3, 7, K, V, V + K), dev, V)


@pytest.mark.parametrize("K", [1, 9])
@pytest.mark.parametrize("V,padded", [(300, 301), (1001, 1008), (4096, 4104), (2047, 2048)])
def test_backward_of_strided_logits(dev, V, padded, K):
    # The columns of a padded vocabulary, rows and columns offset by one element,
    # and a slice of positions: the gradient is contiguous, the logits are not.
    g = torch.Generator().manual_seed(padded)
    full = torch.randn(3, 9, padded, generator=g).mul_(2.0).to(torch.bfloat16).to(dev)
    for zd in (full[..., :V], full[:, 1:8, padded - V:], full[1:, 2:, :V]):
        _check_backward(zd, _ids(zd.shape[0], zd.shape[1], K, V, V + K), dev, V)


def test_backward_of_more_elements_than_one_launch_takes(dev):
    from meshy_amd import logprob, workloads

    T, V = 65536 + 24, 131072 + 1  # past 2^33 elements, in rows that are not 16-byte aligned
    z = workloads.synth_logits(T, V, seed=5, device=dev).unsqueeze(0).requires_grad_(True)
    g = torch.Generator().manual_seed(1)
    y = torch.randint(0, V, (1, T), generator=g)
    grad_out = torch.randn(1, T, generator=g)
    lp = logprob.logprobs_and_entropy(z, y.to(dev))
    grad, = torch.autograd.grad(lp, z, grad_out.to(dev))
    step = 2 ** 33 // V // 8 * 8  # rows of the first launch
    rows = torch.tensor([0, 1, step - 1, step, step + 1, T - 1])
    ref = _grad_ref(z[0, rows].detach().cpu(), y[0, rows, None], grad_out[0, rows, None],
                    logprob.logsumexp_rows(z.detach()[:, rows])[0].cpu())
    err = (grad[0, rows].cpu().double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-5).all()
