"""The K-loop contrastive forward (rows wider than the tiled kernel's, fp32):
remainders of slices, chunks and four-tile steps, query blocks across waves,
documents by rank, dealt and contiguous, unaligned rows through the workspace
copy, invalid documents; and the bits of the pair kernels, and of the route
without a workspace."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import maxsim_amd
from maxsim_amd._ops import ops
from oracle import maxsim_oracle as oracle

from ._helpers import (KLOOP, KLOOP_WS, PAIR, SCORE_TOL, assert_close, check_argmax,
                       contrastive_c_abi, contrastive_pair_kernels, contrastive_route,
                       make_contrastive, np64, npi, one_element_off)

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _check(q, d, off, scores, argmax):
    qn, dn, on = np64(q), np64(d), npi(off)
    s_ref, a_ref = oracle.contrastive_forward(qn, dn, on)
    assert_close(scores, s_ref, **SCORE_TOL[q.dtype])
    check_argmax(npi(argmax), a_ref, lambda i: qn[i[0], i[2]], lambda i, j: dn[on[i[1]] + j])


@pytest.mark.parametrize("Nq,Lq,dim,d_lens,dtype", [
    (130, 32, 80, [1, 32, 33, 128, 129, 40], BF16),      # one slice and one chunk
    (101, 31, 96, [64] * 3 + [1] * 5, F16),
    (257, 20, 256, [200, 97, 31], BF16),
    (17, 32, 768, [5, 160], BF16),
    (129, 33, 144, [300, 1, 129], F16),                   # blocks across waves
    (3, 200, 160, [70, 33], BF16),                        # 7 of 8 blocks
    (1, 256, 160, [70, 33], BF16),                        # all 8
    (1, 257, 160, [70, 33], BF16),                        # one more than a workgroup holds
    (769, 32, 128, [128, 1, 31, 96], F32),
    (513, 40, 48, [33, 64, 2], F32),
    (5, 130, 384, [50, 9], F32),                          # five blocks
    (5, 32, 300, [33, 64, 2, 129], BF16),                 # rows that are copied
    (86, 70, 100, [33, 64, 2], F16),
    (257, 9, 101, [33, 64, 2], BF16),
    (1025, 9, 67, [33, 64, 2], F32),
])
def test_kloop_forward(Nq, Lq, dim, d_lens, dtype):
    q, d, off = make_contrastive(Nq, Lq, dim, d_lens, dtype, seed=dim, unit=True)
    assert contrastive_route(q, d, off) in ((KLOOP, KLOOP_WS) if Lq <= 256 else (PAIR,))
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    _check(q, d, off, scores, argmax)
    assert torch.equal(maxsim_amd.score_contrastive(q, d, off), scores)
    for s, a in (contrastive_c_abi(q, d, off), contrastive_pair_kernels(q, d, off)):
        assert torch.equal(s, scores) and torch.equal(a, argmax)


# documents: one per workgroup with all resident (long and short paired) and in
# several rounds, dealt, and in contiguous runs; the last also puts the
# queries' fragments in order
@pytest.mark.parametrize("Nq,Lq,Nb,dim", [(40, 32, 64, 96), (70, 32, 72, 96), (300, 32, 40, 96),
                                          (64, 32, 250, 80), (200, 32, 700, 144)])
def test_kloop_document_chunks(Nq, Lq, Nb, dim):
    gen = torch.Generator().manual_seed(Nb)
    d_lens = torch.randint(1, 150, (Nb,), generator=gen).tolist()
    q, d, off = make_contrastive(Nq, Lq, dim, d_lens, BF16, seed=Nq, unit=True)
    assert contrastive_route(q, d, off) in (KLOOP, KLOOP_WS)
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    sim = (q.float().view(Nq * Lq, dim) @ d.float().T).view(Nq, Lq, -1)
    ends = off.tolist()
    for b in range(Nb):
        m, a = sim[:, :, ends[b]:ends[b + 1]].max(dim=-1)
        torch.testing.assert_close(scores[:, b], m.sum(1), **SCORE_TOL[BF16])
        # products in another order: near ties may differ (about one in 10^5)
        assert float((argmax[:, b] != a).float().mean()) < 1e-3
    for s, am in (contrastive_c_abi(q, d, off), contrastive_pair_kernels(q, d, off)):
        assert torch.equal(s, scores) and torch.equal(am, argmax)


@pytest.mark.parametrize("dim", [96, 100])
def test_kloop_misaligned_rows_and_invalid_documents(dim):
    q, d, off = make_contrastive(160, 32, dim, [20, 40, 10, 33, 50], BF16, seed=3, unit=True)
    good, good_am = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    assert contrastive_route(q, one_element_off(d), off) == KLOOP_WS  # 2-byte boundary
    scores, argmax = ops.maxsim_contrastive_forward_with_argmax(q, one_element_off(d), off)
    assert torch.equal(scores, good) and torch.equal(argmax, good_am)
    bad = off.clone()
    bad[2] = bad[3]  # document 2 is empty, document 1 longer
    scores, argmax = ops.maxsim_contrastive_forward_with_argmax(q, d, bad)
    assert bool(torch.isnan(scores[:, 2]).all()) and not bool(argmax[:, 2].any())
    keep = [0, 3, 4]
    assert torch.equal(scores[:, keep], good[:, keep])
    assert torch.equal(argmax[:, keep], good_am[:, keep])


@pytest.mark.parametrize("dim", [96, 100])
def test_kloop_nan_and_infinity(dim):
    """NaN and infinite rows against the oracle: a NaN similarity never wins, a
    token whose similarities are all NaN contributes -inf and argmax 0."""
    q, d, off = make_contrastive(260, 32, dim, [40, 33, 70], BF16, seed=5, unit=True)
    d[3, 7] = float("nan")
    d[45, 95] = float("inf")
    d[80, 0] = float("-inf")
    q[1, 4] = float("nan")
    q[2, :, 0] = 0  # 0 * -inf
    assert contrastive_route(q, d, off) in (KLOOP, KLOOP_WS)
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    with np.errstate(invalid="ignore"):
        s_ref, a_ref = oracle.contrastive_forward(np64(q), np64(d), npi(off))
    s, a = scores.double().cpu().numpy(), npi(argmax)
    finite = np.isfinite(s_ref)
    assert np.isneginf(s_ref[1, 0]) and np.isposinf(s_ref[0, 1])
    assert np.array_equal(s[~finite], s_ref[~finite], equal_nan=True)  # inf - inf among them
    assert_close(torch.from_numpy(s[finite]), s_ref[finite], **SCORE_TOL[BF16])
    # near ties of finite similarities may differ (about one in 10^5)
    assert (a != a_ref).mean() < 1e-4 and not a[1, :, 4].any()
    pair_s, pair_a = contrastive_pair_kernels(q, d, off)
    torch.testing.assert_close(pair_s, scores, rtol=0, atol=0, equal_nan=True)
    assert torch.equal(pair_a, argmax)


def test_kloop_without_room_for_the_workspace():
    """Where the device has no room for the workspace, the forward runs on the
    kernels that need none, with the same bits."""
    q, d, off = make_contrastive(16, 32, 100, [130] * 10000, BF16, seed=9, unit=True)
    assert contrastive_route(q, d, off) == KLOOP_WS
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info(q.device)[1]
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
    held = []
    try:
        # fill what is left, in the cached segments too; then make room for the
        # outputs (20 MB), not for the copy (290 MB)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(48 << 20, dtype=torch.uint8, device=q.device))
        held.pop()
        got, got_am = maxsim_amd.score_contrastive_with_argmax(q, d, off)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(200 << 20, dtype=torch.uint8, device=q.device)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, scores) and torch.equal(got_am, argmax)
