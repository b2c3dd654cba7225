"""The backward of short rows, and of rows that are not contiguous.

Waves take 8 to 64 whole rows (those of fewer than 256 logits with one id, and
of fewer than 512 with 2 to 16 ids from 8193 rows on), so the sizes lie around the
rows per wave (V = 16, 32, 64, 128 halve them), the chunk (V below 8 puts several
rows into one, V % 8 != 0 splits them), and the last wave's rows; longer strided
rows are read with two 16-byte loads where a chunk holds a row's end.
Against float64 with the bounds of test_row_alignment_gpu.
"""
import pytest
import torch

from test_row_alignment_gpu import _check_backward, _ids

pytestmark = pytest.mark.gpu

SHORT = [2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 200, 255]


def _logits(rows, T, V, g, dev):
    return torch.randn(rows, T, V, generator=g).mul_(2.0).to(torch.bfloat16).to(dev)


@pytest.mark.parametrize("K", [1, 2, 9, 65, 256])
@pytest.mark.parametrize("V", SHORT)
def test_contiguous_rows(dev, V, K):
    g = torch.Generator().manual_seed(V)
    for rows, T in ((1, 5), (3, 43), (1, 517)):  # 5 rows: fewer than a wave takes
        _check_backward(_logits(rows, T, V, g, dev), _ids(rows, T, K, V, V + K), dev, V)


@pytest.mark.parametrize("K", [2, 9, 16, 17])
@pytest.mark.parametrize("V", [2, 8, 17, 64, 100, 257, 511])
@pytest.mark.parametrize("n", [8192, 8193])
def test_many_rows_with_several_ids(dev, n, V, K):
    g = torch.Generator().manual_seed(V)
    full = _logits(1, n, V + 1, g, dev)
    _check_backward(full[..., 1:] if K == 9 else full[..., :V].contiguous(), _ids(1, n, K, V, V + K), dev, V)


@pytest.mark.parametrize("n", [40000, 140000, 270000])
def test_more_rows_per_wave(dev, n):
    g = torch.Generator().manual_seed(n)
    _check_backward(_logits(1, n, 3, g, dev), _ids(1, n, 1, 3, n), dev, n)


@pytest.mark.parametrize("K", [1, 9])
@pytest.mark.parametrize("V", SHORT + [256, 257, 263, 264, 511, 512, 1001, 4104])
def test_strided_rows(dev, V, K):
    g = torch.Generator().manual_seed(V)
    full = _logits(3, 47, V + 9, g, dev)
    # Padded columns, an odd start, a slice of positions (rows not evenly apart),
    # every second position, and positions in front of rows.
    for zd in (full[..., :V], full[..., 1:V + 1], full[:, 2:45, 9:], full[:, ::2, 8:V + 8],
               full.transpose(0, 1)[..., :V], full[:1, :1, 3:V + 3]):
        _check_backward(zd, _ids(zd.shape[0], zd.shape[1], K, V, V + K), dev, V)


@pytest.mark.parametrize("V", [3, 8, 200, 257])
def test_contiguous_rows_from_an_odd_element(dev, V):
    g = torch.Generator().manual_seed(V)
    flat = torch.randn(2 * 33 * V + 5, generator=g).to(torch.bfloat16).to(dev)
    for offset in (1, 5):
        zd = flat[offset:offset + 2 * 33 * V].view(2, 33, V)
        _check_backward(zd, _ids(2, 33, 9, V, V), dev, V)
