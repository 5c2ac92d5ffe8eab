"""Padded and packed forwards over embedding widths that are not whole aligned
fragments: every remainder of a row's last 8 elements, rows on any element
boundary, the pair kernels of few and of many pairs, wide rows."""

from __future__ import annotations

import pytest
import torch

import maxsim_amd
from maxsim_amd._ops import ops
from oracle import maxsim_oracle as oracle

from ._helpers import (DTYPES, GRAD_TOL, SCORE_TOL, assert_close, check_argmax, make_packed, make_padded,
                       np64, npi)

pytestmark = pytest.mark.gpu

WIDTHS = [1, 7, 8, 9, 15, 16, 17, 26, 35, 44, 61, 96, 100, 118, 127, 143, 201, 255, 300, 301]


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t).split(".")[-1])
@pytest.mark.parametrize("dim", WIDTHS)
def test_padded_forward_row_widths(dim, dtype):
    q, d, ql, dl = make_padded(3, 5, 35, 40, dim, dtype, seed=dim)
    s, a = maxsim_amd.score_candidates_padded_with_argmax(q, d, ql, dl)
    qn, dn = np64(q), np64(d)
    s_ref, a_ref = oracle.padded_forward(qn, dn, npi(ql), npi(dl))
    # |q||d| grows like sqrt(dim): the absolute floor with it
    tol = dict(SCORE_TOL[dtype], atol=SCORE_TOL[dtype]["atol"] * max(1.0, dim / 64))
    assert_close(s, s_ref, **tol)
    check_argmax(npi(a), a_ref, lambda i: qn[i[0], i[2]], lambda i, j: dn[i[0], i[1], j])
    # rows that start one element off give the same bits
    qs, ds = (torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view_as(t).copy_(t)
              for t in (q, d))
    s2, a2 = maxsim_amd.score_candidates_padded_with_argmax(qs, ds, ql, dl)
    assert torch.equal(s, s2) and torch.equal(a, a2)


@pytest.mark.parametrize("dim,dtype", [(20, torch.bfloat16), (96, torch.float16),
                                       (100, torch.float32), (201, torch.bfloat16),
                                       (300, torch.float16)])
def test_packed_forward_row_widths_many_pairs(dim, dtype):
    """1100 pairs (a wave per pair) against the same pairs in small batches (a
    workgroup per pair), bit for bit, and the last row of the last document at
    the end of its allocation."""
    args = make_packed(20, 60, 1100, dim, (1, 40), (1, 70), dtype, seed=dim)
    q, qo, d, do, qi, di = args
    s, a = ops.maxsim_packed_forward_with_argmax(q, qo, d, do, qi, di, 40)
    for lo in (0, 700):
        s2, a2 = ops.maxsim_packed_forward_with_argmax(q, qo, d, do, qi[lo:lo + 400].contiguous(),
                                                       di[lo:lo + 400].contiguous(), 40)
        assert torch.equal(s[lo:lo + 400], s2) and torch.equal(a[lo:lo + 400], a2)
    s_ref, _ = oracle.packed_forward(np64(q), npi(qo), np64(d), npi(do), npi(qi), npi(di), 40)
    tol = dict(SCORE_TOL[dtype], atol=SCORE_TOL[dtype]["atol"] * max(1.0, dim / 64))
    assert_close(s, s_ref, **tol)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t).split(".")[-1])
@pytest.mark.parametrize("B,C,Lq,Ld,dim", [
    (3, 5, 20, 40, 100), (2, 40, 9, 17, 128), (1, 300, 5, 12, 67), (4, 3, 70, 33, 300),
    (2, 16, 1, 1, 8), (2, 17, 33, 40, 5),
])
def test_padded_backward_row_widths(B, C, Lq, Ld, dim, dtype):
    """Both padded gradients of one launch, fp32 and in the inputs' dtype, with
    one to eight lanes per query row and candidates that are not a multiple of
    the gathers in flight; padding rows are zero."""
    q, d, ql, dl = make_padded(B, C, Lq, Ld, dim, dtype, seed=dim + C)
    _, a = maxsim_amd.score_candidates_padded_with_argmax(q, d, ql, dl)
    g = torch.randn(B, C, generator=torch.Generator().manual_seed(C))
    flat = (g.to(q.device).reshape(-1), q.reshape(B * Lq, dim), d.reshape(B * C * Ld, dim), ql,
            dl.reshape(-1), a, Lq, Ld, C)
    dq, dd = ops.maxsim_padded_backward(*flat)
    dq_ref, dd_ref = oracle.padded_backward(np64(g), np64(q), np64(d), npi(ql), npi(dl), npi(a))
    assert_close(dq.view(q.shape), dq_ref, **GRAD_TOL[dtype])
    assert_close(dd.view(d.shape), dd_ref, **GRAD_TOL[dtype])
    dq16, dd16 = ops.maxsim_padded_backward_typed(*flat)
    assert torch.equal(dq16, dq.to(dtype)) and torch.equal(dd16, dd.to(dtype))


@pytest.mark.parametrize("dtype,B,Ld,dim", [
    (torch.float32, 160, 200, 256),  # whole rows per lane group, fp32
    (torch.bfloat16, 80, 251, 600),  # single elements, 16 bit
    (torch.float16, 80, 251, 601),   # rows on any boundary
])
def test_padded_backward_two_launches(dtype, B, Ld, dim):
    """Gradients beyond the size up to which they share a launch, bit for bit
    those of the batch's halves, which do share one."""
    C, Lq = 13, 20
    q, d, ql, dl = make_padded(B, C, Lq, Ld, dim, dtype, seed=dim)
    limit = (384 if dtype == torch.float32 else 192) << 20
    assert d.numel() * d.element_size() > limit > d.numel() * d.element_size() // 2
    gen = torch.Generator().manual_seed(1)
    a = torch.minimum(torch.randint(0, Ld, (B, C, Lq), generator=gen, dtype=torch.int32).to(q.device),
                      dl[..., None] - 1)
    g = torch.randn(B, C, generator=gen).to(q.device)

    def grads(lo, hi):
        n = hi - lo
        return ops.maxsim_padded_backward_typed(
            g[lo:hi].reshape(-1), q[lo:hi].reshape(n * Lq, dim), d[lo:hi].reshape(n * C * Ld, dim),
            ql[lo:hi], dl[lo:hi].reshape(-1), a[lo:hi].reshape(n * C, Lq), Lq, Ld, C)

    dq, dd = grads(0, B)
    halves = [grads(0, B // 2), grads(B // 2, B)]
    assert torch.equal(dq, torch.cat([h[0] for h in halves]))
    assert torch.equal(dd, torch.cat([h[1] for h in halves]))
