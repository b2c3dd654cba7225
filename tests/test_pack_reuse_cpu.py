"""Batches of one pack_step read after another pack_step on the same samples.

The second step rewrites the pinned plan tables; the first one's batches must
still show the first plan.  The copies and kernels are replaced by stand-ins
that do nothing (the shapes and the attention metadata come from the host), so
that the host path runs on the CPU.
"""
import gc
import weakref

import numpy as np
import pytest
import torch

from meshy_amd import _lib, pipeline
from meshy_amd.plan import PlannerConfig

FIELDS = ("input_ids", "labels", "positions", "mask", "doc_ids", "rollout_logprobs", "advantage_tokens")


class _HostOnly:
    _DEVICE = ("meshy_copy_to_device", "meshy_grpo_advantage", "meshy_pack_micro_batches")

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        return (lambda *a: 0) if name in self._DEVICE else getattr(self._lib, name)


@pytest.fixture
def host_only(monkeypatch):
    lib = _HostOnly(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    monkeypatch.setattr(pipeline.RaggedSamples, "record_copy", lambda self, device: None)


def _ragged(lengths, seed=0):
    rng = np.random.default_rng(seed)
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    n = int(off[-1])
    return pipeline.RaggedSamples.from_arrays(
        rng.integers(0, 1000, n), (rng.random(n) < 0.7).astype(np.float32), rng.random(n).astype(np.float32), off,
        rng.random(len(lengths)), np.arange(0, len(lengths) + 1, 2))


def _cfg(layout, budget):
    return PlannerConfig(layout=layout, mini_batch_size=8, seq_len=256, align=64 if layout == "packed" else 1,
                         max_tokens_per_micro=budget)


def _seen(res):
    """Everything of a result's batches that the host decides."""
    out = []
    for mb in res.batches:
        meta = mb.attention_masks
        out.append(([tuple(getattr(mb, f).shape) for f in FIELDS],
                    [getattr(mb, f).storage_offset() * getattr(mb, f).element_size() for f in FIELDS],
                    tuple(mb.lengths.shape), None if meta is None else (tuple(meta.cu_seq_q.shape), meta.max_q)))
    return out


@pytest.mark.parametrize("layout", ["packed", "padded"])
def test_first_result_read_after_a_second_step(host_only, layout):
    lengths = np.random.default_rng(3).integers(5, 250, 16)
    cpu = torch.device("cpu")
    first, second = _cfg(layout, 512), _cfg(layout, 1024)
    want = _seen(pipeline.pack_step(_ragged(lengths), first, cpu))
    ragged = _ragged(lengths)
    res = pipeline.pack_step(ragged, first, cpu)
    other = pipeline.pack_step(ragged, second, cpu)
    assert _seen(other) != want
    assert _seen(res) == want
    ranks = [pipeline.pack_step(ragged, first, cpu, dp_size=2, rank=r) for r in (0, 1)]
    for r in (0, 1):
        assert _seen(ranks[r]) == _seen(pipeline.pack_step(_ragged(lengths), first, cpu, dp_size=2, rank=r))


def test_staging_buffer_lives_as_long_as_a_batch(host_only):
    # The copies out of the pinned buffer may still be queued when the caller
    # drops the samples.
    ragged = _ragged([10, 20, 30, 40])
    alive = weakref.ref(ragged.buf)
    res = pipeline.pack_step(ragged, _cfg("packed", 512), torch.device("cpu"))
    batch = res.batches[0]
    del ragged, res
    gc.collect()
    assert alive() is not None
    del batch
    gc.collect()
    assert alive() is None


def test_micros_that_do_not_fill_the_outputs_are_refused():
    sizes = np.array([64, 64], np.int64).tobytes()
    ones = np.ones(2, np.int64).tobytes()
    buf = torch.zeros(4096, dtype=torch.uint8)
    views = _lib.stage().token_views
    assert len(views(buf, ((0, 4),), ones, sizes, 128)) == 2
    for elements in (127, 129, 192, 0):
        with pytest.raises(ValueError):
            views(buf, ((0, 4),), ones, sizes, elements)
