"""dQ split by document ranges: the paced fp32 gathers, two and four loads in
flight for 16-bit rows, on either side of each choice, with more documents than
a table holds and remainders everywhere, against 64-bit sums."""

from __future__ import annotations

import pytest
import torch

from maxsim_amd._ops import ops

from ._helpers import DEVICE, offsets_from_lengths

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("dtype,dim,Nq,Lq,Nb", [
    (F32, 64, 55, 32, 600),     # four loads in flight
    (F32, 64, 540, 32, 61),     # queries beyond 4 MiB: paced
    (F32, 128, 33, 32, 1000),
    (F32, 136, 16, 33, 2000),   # paced, more than one table of documents
    (F32, 256, 129, 32, 257),
    (F32, 768, 40, 9, 3001),
    (F32, 2048, 10, 50, 2100),  # one row per workgroup
    (F32, 300, 20, 32, 1701),   # rows on 16 bytes, a part-filled last slice
    (BF16, 384, 130, 32, 257),  # two loads in flight
    (BF16, 264, 130, 33, 255),  # four
    (F16, 768, 61, 64, 300),
])
def test_contrastive_dq_split(dtype, dim, Nq, Lq, Nb):
    assert Nq * Lq * Nb >= 1 << 20  # the split needs this much
    gen = torch.Generator(device=DEVICE).manual_seed(dim + Nb)
    lens = torch.randint(1, 6, (Nb,), generator=gen, device=DEVICE)
    off = offsets_from_lengths(lens.tolist()).to(DEVICE)
    q = torch.randn(Nq, Lq, dim, generator=gen, device=DEVICE).to(dtype)
    d = torch.randn(int(lens.sum()), dim, generator=gen, device=DEVICE).to(dtype)
    g = torch.randn(Nq, Nb, generator=gen, device=DEVICE)
    am = (torch.rand(Nq, Nb, Lq, generator=gen, device=DEVICE) * lens[None, :, None]).int()
    am = torch.minimum(am, lens[None, :, None].int() - 1)
    dq, _ = ops.maxsim_contrastive_backward(g, q, d, off, am)
    want = torch.zeros(Nq, Lq, dim, dtype=torch.float64, device=DEVICE)
    size = torch.zeros_like(want)
    for b, start in enumerate(off.tolist()[:-1]):
        rows = d[start + am[:, b].long()].double()
        term = rows * g[:, b, None, None].double()
        want += term
        size += term.abs()
    # sequential fp32 sums in eight ranges, then the eight: each partial sum
    # rounds by at most 2^-24 of the terms' absolute sum
    bound = size * ((Nb + 7) // 8 + 9) * 2.0 ** -24
    assert bool(((dq.view_as(want).double() - want).abs() <= bound).all())
