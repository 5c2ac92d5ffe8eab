"""Contrastive queries of several 32-token blocks: a query's blocks spread over
the waves of one workgroup, their sums met in LDS (1 to 16 blocks, groups that
the blocks do not fill, more blocks than a workgroup holds, documents that end
at every tile, invalid documents)."""

from __future__ import annotations

import pytest
import torch

import maxsim_amd
from maxsim_amd._ops import ops
from oracle import maxsim_oracle as oracle

from ._helpers import (PAIR, SCORE_TOL, TILED, assert_close, check_argmax,
                       contrastive_pair_kernels, contrastive_route, make_contrastive, np64, npi)

pytestmark = pytest.mark.gpu


def _check(q, d, off, scores, argmax):
    qn, dn, on = np64(q), np64(d), npi(off)
    s_ref, a_ref = oracle.contrastive_forward(qn, dn, on)
    assert_close(scores, s_ref, **SCORE_TOL[q.dtype])
    check_argmax(npi(argmax), a_ref, lambda i: qn[i[0], i[2]], lambda i, j: dn[on[i[1]] + j])


@pytest.mark.parametrize("Nq,Lq,dim,d_lens,dtype", [
    (6, 65, 128, [1] * 9, torch.bfloat16),             # every tile ends a document
    (6, 96, 128, [32, 33, 1, 64, 65, 7, 31], torch.float16),
    (3, 97, 64, [200, 1, 1, 95], torch.bfloat16),
    (4, 250, 32, [33, 64, 2], torch.float16),
    (2, 289, 128, [40, 1, 129], torch.bfloat16),       # one query per workgroup, 10 blocks
    (2, 512, 64, [40, 31], torch.bfloat16),            # all 16 blocks
    (2, 513, 64, [40, 31], torch.bfloat16),            # one more than a workgroup holds
    (60, 70, 64, [50, 3, 32, 99, 1, 33] * 3, torch.float32),  # five queries of three blocks
    (2, 330, 64, [50, 3, 33], torch.float32),
])
def test_contrastive_query_blocks(Nq, Lq, dim, d_lens, dtype):
    q, d, off = make_contrastive(Nq, Lq, dim, d_lens, dtype, seed=Lq, unit=True)
    assert contrastive_route(q, d, off) == (TILED if Lq <= 512 else PAIR)
    scores, argmax = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    _check(q, d, off, scores, argmax)
    assert torch.equal(maxsim_amd.score_contrastive(q, d, off), scores)
    s, a = contrastive_pair_kernels(q, d, off)
    assert torch.equal(s, scores) and torch.equal(a, argmax)


def test_contrastive_query_blocks_invalid_documents():
    q, d, off = make_contrastive(4, 96, 128, [20, 40, 10, 33, 50], torch.bfloat16, seed=3)
    assert contrastive_route(q, d, off) == TILED
    good, good_am = maxsim_amd.score_contrastive_with_argmax(q, d, off)
    bad = off.clone()
    bad[2] = bad[3]  # document 2 is empty, document 1 longer
    scores, argmax = ops.maxsim_contrastive_forward_with_argmax(q, d, bad)
    assert bool(torch.isnan(scores[:, 2]).all()) and not bool(argmax[:, 2].any())
    keep = [0, 3, 4]
    assert torch.equal(scores[:, keep], good[:, keep])
    assert torch.equal(argmax[:, keep], good_am[:, keep])
