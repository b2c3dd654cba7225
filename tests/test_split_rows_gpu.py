"""Few rows, each divided over several workgroups (up to 128 rows, 49152 logits and more): the rule's edges, rows that
start anywhere, special values, polls that run out, and graph replays (which are not divided)."""
import pytest
import torch

from meshy_amd import _lib
from meshy_amd.logprob import logprobs_and_entropy
from meshy_amd.topk import gather_logprobs

pytestmark = pytest.mark.gpu

# A lane adds at most about 50 exponentials one after the other and 9 merges follow, each 2^-24 off relatively: the sum
# is within 4e-6, the log-sum-exp (below 32, half an ulp 1e-6) within 6e-6.  The entropy divides by that sum a weighted
# sum of terms up to log2 V + 8 < 26.
LOGP_ATOL, ENT_ATOL = 1e-5, 1e-4


def _logits(n, V, seed, offset=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    flat = torch.randn(offset + n * V, generator=gen, device="cuda").mul_(2.0).to(torch.bfloat16)
    labels = torch.randint(V, (1, n), generator=gen, device="cuda")
    return flat[offset:].view(1, n, V), labels


def _exact(logits, ids):
    lp = torch.log_softmax(logits.double(), -1)
    return lp.gather(-1, ids), -(lp.exp() * lp).sum(-1)


def _check(logits, labels, logp, ent):
    want, want_ent = _exact(logits, labels.unsqueeze(-1))
    torch.testing.assert_close(logp.double(), want.squeeze(-1), rtol=0, atol=LOGP_ATOL)
    torch.testing.assert_close(ent.double(), want_ent, rtol=0, atol=ENT_ATOL)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 37, 85, 86, 127, 128, 129])
@pytest.mark.parametrize("V", [49151, 49152, 49153, 65541, 151936])
def test_rows_and_vocabularies(n, V):
    logits, labels = _logits(n, V, n + V)
    _check(logits, labels, *logprobs_and_entropy(logits, labels, with_entropy=True))


@pytest.mark.parametrize("offset", [1, 7, 63])
def test_rows_start_anywhere(offset):
    logits, labels = _logits(5, 50257, offset, offset)
    _check(logits, labels, *logprobs_and_entropy(logits, labels, with_entropy=True))
    strided = logits[:, ::2]
    _check(strided, labels[:, ::2], *logprobs_and_entropy(strided, labels[:, ::2], with_entropy=True))


def test_gathered_ids_in_every_part():
    logits, _ = _logits(7, 131072, 3)
    ids = (torch.arange(64, device="cuda") * 2048 + 2047).expand(1, 7, 64).contiguous()
    got = gather_logprobs(logits, ids)
    torch.testing.assert_close(got.double(), _exact(logits, ids)[0], rtol=0, atol=LOGP_ATOL)


def test_special_values_and_labels():
    V = 131072
    logits, labels = _logits(8, V, 4)
    logits[0, 0, V - 5] = float("nan")      # in the last part
    logits[0, 1, 3] = float("nan")          # in the first
    logits[0, 2, :-1] = float("-inf")       # all but one logit
    logits[0, 3, 70000] = 200.0             # far above the others, in a middle part
    labels[0, 2] = V - 1
    labels[0, 3] = 70000
    labels[0, 4] = -100
    labels[0, 5] = V
    logp = logprobs_and_entropy(logits, labels)[0]
    assert logp[:2].isnan().all() and logp[5].isnan()
    assert logp[4] == 0
    assert logp[2:4].abs().max() <= 1e-4  # one logit has all the weight; 200 log2 e rounds to 1.5e-5
    rest = logits[:, 6:]
    torch.testing.assert_close(logp[6:].double(), _exact(rest, labels[:, 6:].unsqueeze(-1))[0][0, :, 0], rtol=0,
                               atol=LOGP_ATOL)


@pytest.mark.parametrize("n", [1, 37, 128])
def test_polls_that_run_out(n):
    logits, labels = _logits(n, 151936, n)
    logp, ent = torch.empty(2, 1, n, device="cuda").unbind()
    rc = _lib.load().meshy_logprob_entropy_fwd_polls(
        logits.data_ptr(), 1, n, 151936, logits.stride(0), logits.stride(1), labels.data_ptr(), logp.data_ptr(),
        ent.data_ptr(), None, 0, _lib.stream_of(logits.device))
    _lib.check(rc, "meshy_logprob_entropy_fwd_polls")
    _check(logits, labels, logp, ent)


@pytest.mark.parametrize("n", [1, 16, 37, 127])
@pytest.mark.parametrize("V", [49153, 151936])
def test_outputs_do_not_depend_on_who_took_the_parts(n, V):
    # max_polls = 0: the last part's workgroup does not look and takes every part.
    lib, stream = _lib.load(), _lib.stream_of(torch.device("cuda:0"))
    logits, labels = _logits(n, V, n + V + 1, offset=3)
    ids = torch.randint(V, (1, n, 9), device="cuda")
    shape = (logits.data_ptr(), 1, n, V, logits.stride(0), logits.stride(1))
    results = []
    for polls in (4000, 0, 1):
        logp, ent, lse, lse_of_gather = torch.empty(4, 1, n, device="cuda").unbind()
        out = torch.empty(1, n, 9, device="cuda")
        _lib.check(lib.meshy_logprob_entropy_fwd_polls(*shape, labels.data_ptr(), logp.data_ptr(), ent.data_ptr(),
                                                       lse.data_ptr(), polls, stream), "entropy")
        _lib.check(lib.meshy_gather_logprobs_fwd_polls(*shape, ids.data_ptr(), 9, out.data_ptr(),
                                                       lse_of_gather.data_ptr(), polls, stream), "gather")
        results.append((logp, ent, lse, lse_of_gather, out))
    _check(logits, labels, logp, ent)
    torch.testing.assert_close(out.double(), _exact(logits, ids)[0], rtol=0, atol=LOGP_ATOL)
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    eager = logprobs_and_entropy(logits, labels, with_entropy=True)
    assert torch.equal(eager[0], logp) and torch.equal(eager[1], ent)


def test_calls_on_two_streams():
    logits, labels = _logits(37, 151936, 9)
    first = logprobs_and_entropy(logits, labels, with_entropy=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    outs = []
    for _ in range(100):  # more calls than there are ring entries
        outs.append(logprobs_and_entropy(logits, labels, with_entropy=True))
        with torch.cuda.stream(side):
            outs.append(logprobs_and_entropy(logits, labels, with_entropy=True))
    torch.cuda.synchronize()
    for logp, ent in outs:
        torch.testing.assert_close(logp, first[0], rtol=0, atol=LOGP_ATOL)
        torch.testing.assert_close(ent, first[1], rtol=0, atol=ENT_ATOL)


def test_replays_of_a_captured_call_follow_their_inputs():
    logits, labels = _logits(37, 151936, 11)
    logprobs_and_entropy(logits, labels, with_entropy=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logp, ent = logprobs_and_entropy(logits, labels, with_entropy=True)
    for seed in range(3):
        logits.copy_(_logits(37, 151936, 20 + seed)[0])
        graph.replay()
        torch.cuda.synchronize()
        _check(logits, labels, logp, ent)
        logprobs_and_entropy(logits, labels, with_entropy=True)
        torch.cuda.synchronize()
