"""The device-side layout check behind the Python functions: every array kind
and index type, one to 87 workgroups (of at most 128), a bad value at either
end, on workgroup boundaries and in each array, the longest segment, the
reference's errors, and the check's result under capture, tracing and when it
is dropped."""

from __future__ import annotations

import pytest
import torch

import maxsim_amd
from maxsim_amd._ops import ops

from ._helpers import DEVICE, make_contrastive, make_packed, make_padded

pytestmark = pytest.mark.gpu


def _found(status, like):
    return ops.maxsim_check_wait(status, like)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", [1, 2, 1024, 8192, 8193, 70001, 700001])
def test_check_lengths_and_ids(n, dtype):
    gen = torch.Generator().manual_seed(n)
    dlen = torch.randint(1, 51, (n,), generator=gen, dtype=dtype).to(DEVICE)
    qlen = torch.tensor([7], dtype=dtype, device=DEVICE)
    assert _found(ops.maxsim_check_padded(qlen, dlen, 7, 50), qlen) == 0
    assert _found(ops.maxsim_check_padded(qlen, dlen, 6, 50), qlen) == -1
    for at in {0, n // 2, n - 1}:
        for value in (0, 51, -1, 2 ** 31 - 1):
            bad = dlen.clone()
            bad[at] = value
            assert _found(ops.maxsim_check_padded(qlen, bad, 7, 50), qlen) == -1
    if dtype == torch.int64:
        bad = dlen.clone()
        bad[n - 1] = 2 ** 32 + 1  # 1 if narrowed
        assert _found(ops.maxsim_check_padded(qlen, bad, 7, 50), qlen) == -1
    # not contiguous
    wide = torch.zeros(n, 2, dtype=dtype, device=DEVICE)
    wide[:, 0] = dlen
    assert _found(ops.maxsim_check_padded(qlen, wide[:, 0], 7, 50), qlen) == 0


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", [1, 2, 1023, 8191, 8192, 100000])
def test_check_offsets(n, dtype):
    gen = torch.Generator().manual_seed(n)
    lens = torch.randint(1, 9, (n,), generator=gen)
    lens[n // 2] = 11
    off = torch.zeros(n + 1, dtype=dtype)
    off[1:] = lens.cumsum(0)
    total = int(off[-1])
    off = off.to(DEVICE)
    assert _found(ops.maxsim_check_contrastive(off, total, None), off) == 11
    assert _found(ops.maxsim_check_contrastive(off, total + 1, None), off) == -1
    for at in {0, 1, n // 2, n}:
        bad = off.clone()
        bad[at] = total + 5 if at == 0 else off[at - 1]
        assert _found(ops.maxsim_check_contrastive(bad, total, None), off) == -1
    targets = torch.tensor([0, n - 1], device=DEVICE)
    assert _found(ops.maxsim_check_contrastive(off, total, targets), off) == 11
    assert _found(ops.maxsim_check_contrastive(off, total, targets + 1), off) == -1
    one = off[:1].contiguous()
    assert _found(ops.maxsim_check_contrastive(one, 0, None), off) == -1


def test_check_packed_arrays_and_errors():
    args = list(make_packed(6, 9, 40, 32, (1, 12), (1, 20), torch.float16, seed=1))
    q, qo, d, do, qi, di = args
    longest = int((qo[1:] - qo[:-1]).max())
    status = ops.maxsim_check_packed(qo, do, qi, di, q.shape[0], d.shape[0])
    assert _found(status, qo) == longest
    scores, argmax = maxsim_amd.score_pairs_packed_with_argmax(*args)
    assert tuple(argmax.shape) == (40, longest)
    assert torch.equal(maxsim_amd.score_pairs_packed(*args), scores)
    for which, value, word in [(1, -1, "query_offsets"), (3, -1, "document_offsets"),
                               (4, 6, "pair_query_ids"), (5, 9, "pair_document_ids")]:
        bad = [t.clone() for t in args]
        bad[which][-1] = value
        for kw in ({}, {"max_q_len": longest}):
            with pytest.raises(RuntimeError, match=word):
                maxsim_amd.score_pairs_packed_with_argmax(*bad, **kw)
            with pytest.raises(RuntimeError, match=word):
                maxsim_amd.score_pairs_packed(*bad, **kw)
    with pytest.raises(ValueError, match="max_q_len"):
        maxsim_amd.score_pairs_packed(*args, max_q_len=longest - 1)
    torch.cuda.synchronize()


def test_check_waits_when_the_launch_raises():
    """A launch that fails leaves no check writing into a freed buffer: the
    next calls, which reuse it, see their own verdicts."""
    q, d, ql, dl = make_padded(2, 3, 4, 8, 16, torch.float32, seed=2)
    for _ in range(3):
        with pytest.raises(RuntimeError, match="launch failed"):
            status = ops.maxsim_check_padded(ql, dl, 4, 8)

            def launch():
                raise RuntimeError("launch failed")

            maxsim_amd._run_checked(status, ql, launch)
        bad = dl.clone()
        bad[1, 2] = 9
        with pytest.raises(ValueError, match="doc_lengths"):
            maxsim_amd.score_candidates_padded(q, d, ql, bad)
        maxsim_amd.score_candidates_padded(q, d, ql, dl)


def test_check_is_refused_under_capture():
    """With the checks on, a call inside a graph capture raises before anything
    is recorded; the capture, later calls and a capture without the checks are
    not affected."""
    q, d, ql, dl = make_padded(2, 3, 4, 8, 16, torch.float32, seed=5)
    want = maxsim_amd.score_candidates_padded(q, d, ql, dl)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    doubled = torch.empty_like(want)
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captured"):
            maxsim_amd.score_candidates_padded(q, d, ql, dl)
        torch.add(want, want, out=doubled)
    graph.replay()
    assert torch.equal(doubled, 2 * want)
    assert torch.equal(maxsim_amd.score_candidates_padded(q, d, ql, dl), want)


def test_dropped_check_keeps_its_words_until_it_has_run():
    """A check's result dropped while the check still waits in the stream: its
    pinned words are not handed out again before the check has written them."""
    n = 4096
    off = torch.arange(n + 1, dtype=torch.int32, device=DEVICE)
    a = torch.randn(4096, 4096, device=DEVICE)
    torch.cuda.synchronize()
    for _ in range(20):  # tens of milliseconds of work ahead of the check
        a = (a @ a).clamp_(-1, 1)
    busy = torch.cuda.Event()
    busy.record()
    status = ops.maxsim_check_contrastive(off, n, None)
    at = status.data_ptr()
    del status
    others = [torch.zeros(m, dtype=torch.int64).pin_memory() for m in (3, 4, 5, 6, 7, 8, 16)
              for _ in range(8)]
    assert not busy.query(), "the work ahead ended too early for the test to say anything"
    assert at not in {t.data_ptr() for t in others}
    torch.cuda.synchronize()
    assert not any(bool(t.any()) for t in others)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_jit_trace_of_the_checked_functions():
    """torch.jit.trace records the scoring operators with the host checks on
    (the checks themselves stay out of the graph); the traced function scores
    other inputs of the same shapes."""
    q, d, off = make_contrastive(3, 8, 32, [5, 9, 7], torch.float32, seed=1)
    pq, pd, ql, dl = make_padded(2, 3, 4, 8, 16, torch.float32, seed=2)
    packed = make_packed(3, 4, 6, 32, (4, 12), (5, 20), torch.float32, seed=3)
    for fn, args in [(maxsim_amd.score_contrastive, (q, d, off)),
                     (maxsim_amd.score_contrastive_with_argmax, (q, d, off)),
                     (maxsim_amd.score_candidates_padded, (pq, pd, ql, dl)),
                     (maxsim_amd.score_pairs_packed, tuple(packed))]:
        traced = torch.jit.trace(fn, args)
        assert "maxsim_check" not in str(traced.graph)
        other = (torch.flip(args[0], (-1,)), *args[1:])
        for a in (args, other):
            got, want = traced(*a), fn(*a)
            for g, w in zip(got if isinstance(got, tuple) else (got,),
                            want if isinstance(want, tuple) else (want,)):
                assert torch.equal(g, w)
