"""teacher_topk on rows that leave the common path of its buffers.

The kernel buffers the chunks that reach a threshold and compacts a full
buffer, bounds what it lists at the end, and trims ties at the bound.  The rows
below overflow the buffers (ascending, equal and coarse values), tie at the
bound across waves, hide the best values at the row's ends or before a run of
-inf, and start at any element; sizes lie on both sides of each rule on K, the
row's length and the number of rows.  Ids must equal a stable descending
sort's; log-probs lie within 2e-5 of float64 (the log-sum-exp is at most 32 in
magnitude, where fp32 values are 2e-6 apart; its sum adds a few 1e-7 relative).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = ("random", "ascending", "descending", "equal", "coarse", "ends", "prefix", "two_values", "nan")


def _row(kind, V, g):
    z = torch.randn(V, generator=g) * 2.0
    if kind == "ascending":
        z = z.sort().values
    elif kind == "descending":
        z = z.sort(descending=True).values
    elif kind == "equal":
        z = torch.full((V,), -1.5)
    elif kind == "coarse":
        z = z.round()
    elif kind == "ends":
        z[:9] = 20.0
        z[-9:] = 20.0
    elif kind == "prefix":
        z[: (3 * V) // 4] = -float("inf")
    elif kind == "two_values":
        z = (torch.rand(V, generator=g) < 0.5).float()
    elif kind == "nan":
        z[torch.randint(0, V, (3,), generator=g)] = float("nan")
        z[V // 2] = float("inf")
    return z


def _check(zd, k, what, every=1):
    from meshy_amd import topk

    ids, lps = (x[:, ::every] for x in topk.teacher_topk(zd, k))
    z = zd[:, ::every].cpu().double()
    ref = torch.sort(z, dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu(), ref.indices[..., :k]), what
    want = ref.values[..., :k] - torch.logsumexp(z, -1, keepdim=True)
    got = lps.cpu().double()
    assert torch.equal(got.isnan(), want.isnan()), what
    finite = want.isfinite()
    assert torch.equal(got[~finite & ~want.isnan()], want[~finite & ~want.isnan()]), what
    assert (got[finite] - want[finite]).abs().max().item() <= 2e-5 if finite.any() else True, what


@pytest.mark.parametrize("k", [1, 8, 32, 33, 64])
@pytest.mark.parametrize("V,offset", [(64, 0), (71, 3), (1031, 1), (8192, 0), (16387, 63), (50257, 5), (65537, 8),
                                      (131072, 0)])
def test_topk_of_rows_off_the_common_path(dev, V, offset, k):
    g = torch.Generator().manual_seed(V + offset)
    flat = torch.cat([torch.zeros(offset)] + [_row(kind, V, g) for kind in KINDS]).to(torch.bfloat16).to(dev)
    _check(flat[offset:].view(1, len(KINDS), V), min(k, V), f"V={V} offset={offset} k={k}")


# More rows than 256 take smaller workgroups; 2048 rows of more than 65536
# columns have twice the loads in flight.
@pytest.mark.parametrize("k", [5, 64])
@pytest.mark.parametrize("rows,V", [(256, 2049), (257, 2049), (256, 65537), (300, 65537), (2047, 65537), (2048, 65536),
                                    (2048, 65537)])
def test_topk_on_both_sides_of_the_launch_rules(dev, rows, V, k):
    g = torch.Generator(device=dev).manual_seed(rows + V)
    z = torch.randn(1, rows, V, generator=g, device=dev, dtype=torch.bfloat16).mul_(2.0)
    z[:, ::3] = z[:, ::3].sort(dim=-1).values
    z[:, 1::3] = z[:, 1::3].round()
    _check(z, k, f"rows={rows} V={V} k={k}", every=max(1, rows // 40))
