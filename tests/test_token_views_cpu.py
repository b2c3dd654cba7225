"""The native per-token views of a pack launch against slices of its buffer."""
import numpy as np
import pytest
import torch

from meshy_amd import _lib
from meshy_amd.batch import _SCALAR_TYPE

DTYPES = (torch.int64, torch.int32, torch.float32)


def _views(buf, specs, rows, seq):
    return _lib.stage().token_views(buf, specs, np.asarray(rows, np.int64).tobytes(), np.asarray(seq, np.int64).tobytes())


@pytest.mark.parametrize("rows,seq", [([1], [1]), ([1, 1, 1], [64, 2048, 7]), ([3, 1, 2], [5, 0, 9]), ([], [])])
def test_views_are_the_slices(rows, seq):
    sizes = [r * s for r, s in zip(rows, seq)]
    total = sum(sizes)
    buf = torch.from_numpy(np.random.default_rng(len(rows)).integers(0, 256, 3 * (8 * total + 256), dtype=np.uint8))
    at = [k * (8 * total + 255) // 256 * 256 for k in range(3)]
    specs = tuple((o, _SCALAR_TYPE[d]) for o, d in zip(at, DTYPES)) + (None,)
    got = _views(buf, specs, rows, seq)
    assert len(got) == len(rows)
    first = 0
    for micro, r, s in zip(got, rows, seq):
        assert len(micro) == 4 and micro[3] is None
        for t, o, d in zip(micro, at, DTYPES):
            want = buf[o + first * d.itemsize:o + (first + r * s) * d.itemsize].view(d).view(r, s)
            assert t.dtype == d and t.shape == want.shape and t.stride() == want.stride() and t.is_contiguous()
            assert torch.equal(t.view(torch.uint8), want.view(torch.uint8))
            if t.numel():
                assert t.data_ptr() == want.data_ptr()
        first += r * s


def test_storage_and_version_are_the_buffers():
    buf = torch.zeros(512, dtype=torch.uint8)
    (t, u), = _views(buf, ((0, _SCALAR_TYPE[torch.float32]), (256, _SCALAR_TYPE[torch.int64])), [1], [32])
    before = buf._version
    t.add_(1)  # any output's change is seen at the buffer and the other outputs
    assert buf._version == u._version == before + 1
    assert torch.equal(buf[:128].view(torch.float32), torch.ones(32))
    address = u.data_ptr()
    del buf, t
    assert u.sum() == 0 and u.data_ptr() == address  # the storage outlives the buffer


@pytest.mark.parametrize("specs,rows,seq", [
    (((0, 4),), [1], [65]),        # one element past the end
    (((-8, 4),), [1], [1]),
    (((4, 4),), [1], [1]),         # not aligned
    (((0, 999),), [1], [1]),       # no such type
    (((0, 4),), [1, 1], [1]),      # sizes of different lengths
    (((0, 4),), [-1], [1]),
])
def test_bad_regions_are_refused(specs, rows, seq):
    with pytest.raises(ValueError):
        _views(torch.zeros(512, dtype=torch.uint8), specs, rows, seq)


def test_bad_arguments_are_refused():
    with pytest.raises(TypeError):
        _views(torch.zeros(64, dtype=torch.uint8), (7,), [1], [1])
    with pytest.raises(TypeError):
        _views(np.zeros(64, np.uint8), ((0, 4),), [1], [1])
    with pytest.raises(ValueError):
        _views(torch.zeros(64), ((0, 4),), [1], [1])


@pytest.mark.parametrize("made_in", [False, True])
@pytest.mark.parametrize("read_in", [False, True])
def test_views_are_of_the_buffers_kind_whatever_the_mode(made_in, read_in):
    with torch.inference_mode(made_in):
        buf = torch.zeros(512, dtype=torch.uint8)
    with torch.inference_mode(read_in):
        (t, u), = _views(buf, ((0, _SCALAR_TYPE[torch.float32]), (256, _SCALAR_TYPE[torch.int64])), [1], [32])
    assert t.is_inference() == u.is_inference() == made_in
    if not made_in:  # read while scoring, trained on later
        before = buf._version
        t.add_(1)
        assert buf._version == u._version == before + 1
        w = torch.ones(1, 32, requires_grad=True)
        (w * t).sum().backward()
        assert torch.equal(w.grad, torch.ones(1, 32))
