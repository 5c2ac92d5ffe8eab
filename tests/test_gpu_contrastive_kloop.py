"""The K-loop contrastive forward (rows wider than the tiled kernel's, fp32):
remainders of slices, chunks and four-tile steps, query blocks across waves,
documents by rank, dealt and contiguous, unaligned rows through the workspace
copy, invalid documents; and the same bits as the route without a workspace."""

from __future__ import annotations

import ctypes

import pytest
import torch

import maxsim_amd
from maxsim_amd._ops import NATIVE_LIB, ops
from oracle import maxsim_oracle as oracle

from ._helpers import SCORE_TOL, assert_close, check_argmax, make_contrastive, np64, npi

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _check(q, d, off, scores, argmax):
    qn, dn, on = np64(q), np64(d), npi(off)
    s_ref, a_ref = oracle.contrastive_forward(qn, dn, on)
    assert_close(scores, s_ref, **SCORE_TOL[q.dtype])
    check_argmax(npi(argmax), a_ref, lambda i: qn[i[0], i[2]], lambda i, j: dn[on[i[1]] + j])


def _without_workspace(q, d, off):
    """Scores and argmax of the C ABI entry point, which takes no workspace."""
    P, I64 = ctypes.c_void_p, ctypes.c_int64
    fn = ctypes.CDLL(str(NATIVE_LIB)).maxsim_amd_contrastive_forward_with_argmax
    fn.argtypes = [ctypes.c_int, P, I64, I64, P, I64, P, I64, I64, P, P, P]
    nq, lq, dim = q.shape
    nb = off.numel() - 1
    s = torch.empty(nq, nb, device=q.device)
    a = torch.empty(nq, nb, lq, dtype=torch.int32, device=q.device)
    dt = {F32: 0, F16: 1, BF16: 2}[q.dtype]
    assert fn(dt, q.data_ptr(), nq, lq, d.data_ptr(), d.shape[0], off.data_ptr(), nb, dim,
              s.data_ptr(), a.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    return s, a


# enough pairs for the K-loop kernel: Nq * documents * blocks >= 768 (16-bit rows
# up to 256), 3072 (fp32)
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
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    _check(q, d, off, scores, argmax)
    assert torch.equal(maxsim_amd.score_contrastive(q, d, off), scores)
    s, a = _without_workspace(q, d, off)
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
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    sim = torch.einsum("qid,td->qit", q.float(), d.float())
    for b in (0, 1, Nb // 2, Nb - 1):
        m, a = sim[:, :, int(off[b]):int(off[b + 1])].max(dim=-1)
        torch.testing.assert_close(scores[:, b], m.sum(1), **SCORE_TOL[BF16])
        assert float((argmax[:, b] != a).float().mean()) < 1e-3
    s, am = _without_workspace(q, d, off)
    assert torch.equal(s, scores) and torch.equal(am, argmax)


@pytest.mark.parametrize("dim", [96, 100])
def test_kloop_misaligned_rows_and_invalid_documents(dim):
    q, d, off = make_contrastive(160, 32, dim, [20, 40, 10, 33, 50], BF16, seed=3, unit=True)
    good, good_am = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    shifted = torch.empty(d.numel() + 1, dtype=d.dtype, device=d.device)[1:].view_as(d)
    shifted.copy_(d)  # rows on a 2-byte boundary
    scores, argmax = ops.maxsim_contrastive_forward_with_argmax(q, shifted, off)
    assert torch.equal(scores, good) and torch.equal(argmax, good_am)
    bad = off.clone()
    bad[2] = bad[3]  # document 2 is empty, document 1 longer
    scores, argmax = ops.maxsim_contrastive_forward_with_argmax(q, d, bad)
    assert bool(torch.isnan(scores[:, 2]).all()) and not bool(argmax[:, 2].any())
    keep = [0, 3, 4]
    assert torch.equal(scores[:, keep], good[:, keep])
    assert torch.equal(argmax[:, keep], good_am[:, keep])


def test_kloop_nan_and_infinity():
    q, d, off = make_contrastive(260, 32, 100, [40, 33, 70], BF16, seed=5, unit=True)
    d[3, 7] = float("nan")
    d[45, 99] = float("inf")
    d[80, 0] = float("-inf")
    q[1, 4] = float("nan")
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    s, a = _without_workspace(q, d, off)
    torch.testing.assert_close(scores, s, rtol=0, atol=0, equal_nan=True)
    assert torch.equal(a, argmax)


def test_kloop_without_room_for_the_workspace():
    """Where the device has no room for the workspace, the forward runs on the
    kernels that need none, with the same bits."""
    torch.cuda.empty_cache()  # the inputs in segments of their own, with nothing free in them
    q, d, off = make_contrastive(16, 32, 100, [130] * 10000, BF16, seed=9, unit=True)
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info(q.device)[1]
    torch.cuda.set_per_process_memory_fraction(
        (torch.cuda.memory_reserved() + (64 << 20)) / total)  # the copy takes 290 MB
    try:
        got, got_am = maxsim_amd.score_contrastive_with_argmax(q, d, off)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(128 << 20, dtype=torch.uint8, device=q.device)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, scores) and torch.equal(got_am, argmax)
