"""Contrastive gradients where the dd kernel splits few documents into parts of
the embedding dimension (even and uneven parts, one slice over, rows of any
width), against the oracle."""

from __future__ import annotations

import pytest
import torch

from maxsim_amd._ops import ops
from oracle import maxsim_oracle as oracle

from ._helpers import GRAD_TOL, assert_close, make_contrastive, np64, npi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Nq,Lq,dim,Nb", [
    (5, 20, 64, 3),       # two parts of four slices
    (5, 20, 72, 3),       # nine slices
    (4, 9, 768, 5),       # eight parts of twelve
    (4, 9, 392, 5),       # 49 slices: the last part is short
    (6, 33, 300, 7),      # rows on 8-byte boundaries
    (3, 7, 131, 4),       # rows on any boundary
    (40, 20, 256, 130),   # parts of at least eight slices
])
def test_contrastive_backward_dimension_parts(Nq, Lq, dim, Nb, dtype):
    gen = torch.Generator().manual_seed(dim)
    d_lens = torch.randint(1, 60, (Nb,), generator=gen).tolist()
    q, d, off = make_contrastive(Nq, Lq, dim, d_lens, dtype, seed=dim, unit=True)
    _, argmax = ops.maxsim_contrastive_forward_with_argmax(q, d, off)
    g = torch.randn(Nq, Nb, generator=gen)
    dq, dd = ops.maxsim_contrastive_backward(g.to(q.device), q, d, off, argmax)
    dq_ref, dd_ref = oracle.contrastive_backward(np64(g), np64(q), np64(d), npi(off), npi(argmax))
    assert_close(dq.view(q.shape), dq_ref, **GRAD_TOL[dtype])
    assert_close(dd, dd_ref, **GRAD_TOL[dtype])
