"""Which kernel the contrastive forward takes (CPU only: the host's rule, no
launch).  The tiled and K-loop kernels multiply every query block of a
workgroup, so batches that leave most of them empty, and long queries with few
pairs, belong to the pair kernels; full ones do not."""

from __future__ import annotations

import ctypes
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "maxsim_amd" / "libmaxsim_amd.so"
F32, F16, BF16 = 0, 1, 2
PAIR, TILED, KLOOP, KLOOP_WS = 0, 1, 2, 3
ROWS = 170  # mean document length


@pytest.fixture(scope="module")
def route():
    fn = ctypes.CDLL(str(LIB)).maxsim_internal_contrastive_route
    I64, P = ctypes.c_int64, ctypes.c_void_p
    fn.argtypes = [ctypes.c_int, P, I64, I64, P, I64, I64, I64]

    def kernel(dtype, dim, nq, lq, nb, q=1 << 20, d=1 << 30):
        return fn(dtype, q, nq, lq, d, nb * ROWS, nb, dim)

    return kernel


@pytest.mark.parametrize("dtype,dim,nq,lq,nb", [
    (F32, 128, 1, 32, 4000),    # 115 us on pair_kernel, 463 on the K-loop kernel
    (F32, 128, 4, 32, 4000),    # 371, 470
    (F32, 128, 9, 32, 4000),    # a second group for one query: 698, 838
    (F32, 128, 5, 77, 1000),    # two queries of three blocks to a group
    (F32, 256, 1, 32, 4000),    # 215, 891
    (F32, 200, 1, 32, 4000),    # 536, 943
    (F32, 384, 1, 32, 4000),    # 519, 1323
    (BF16, 256, 1, 32, 1000),   # 27, 55
    (BF16, 100, 1, 32, 4000),   # a copy of all documents: 36, 128
    (BF16, 100, 4, 32, 400),    # 17, 26
    (BF16, 300, 1, 32, 4000),   # 246, 314
    (F32, 64, 1, 96, 4),        # long queries, one workgroup per document: 126, 482
    (F32, 64, 5, 96, 64),       # 42, 72
    (F32, 64, 1, 77, 1000),     # 76, 203
    (F32, 32, 2, 96, 256),      # 25, 42
    (BF16, 64, 1, 96, 1000),    # 27, 39
    (BF16, 64, 1, 128, 4000),   # 34, 63
    (BF16, 128, 1, 77, 4000),   # 49, 76
    (F16, 32, 1, 96, 500),      # 9, 16
])
def test_unfilled_groups_take_the_pair_kernels(route, dtype, dim, nq, lq, nb):
    assert route(dtype, dim, nq, lq, nb) == PAIR


@pytest.mark.parametrize("dtype,dim,nq,lq,nb,kernel", [
    (F32, 128, 8, 32, 4000, KLOOP),      # 657 us on pair_kernel, 479 on the K-loop kernel
    (F32, 128, 72, 32, 72, KLOOP),
    (F32, 128, 1, 250, 1000, KLOOP),     # 285, 172
    (F32, 72, 6, 32, 4000, KLOOP_WS),    # 540, 391
    (F32, 72, 9, 32, 4000, KLOOP_WS),    # 762, 627
    (F32, 200, 4, 32, 4000, KLOOP_WS),
    (F32, 384, 8, 32, 1000, KLOOP),
    (BF16, 96, 4, 32, 4000, KLOOP_WS),
    (BF16, 256, 4, 32, 1000, KLOOP_WS),  # 65, 51
    (BF16, 100, 8, 32, 4000, KLOOP_WS),  # 201, 130
    (BF16, 300, 2, 32, 4000, KLOOP_WS),  # 462, 317
    (BF16, 300, 1, 32, 100, KLOOP_WS),   # 37, 31
    (BF16, 768, 1, 32, 1000, KLOOP_WS),
    (BF16, 768, 64, 32, 64, KLOOP_WS),
    (BF16, 384, 32, 11, 64, KLOOP),      # queries that fill a third of their blocks
    (BF16, 272, 8, 32, 64, KLOOP),       # 16.7, 18.3 with the queries in order
    (F32, 64, 10, 77, 1000, TILED),      # 456, 353
    (F32, 64, 9, 250, 64, TILED),        # 161, 77
    (BF16, 64, 3, 77, 1000, TILED),      # 51, 39
    (BF16, 64, 1, 250, 64, TILED),       # 27, 14
    (BF16, 128, 1, 96, 256, TILED),
    (BF16, 128, 3, 96, 4000, TILED),     # 129, 77
    (F16, 128, 150, 96, 501, TILED),
    (BF16, 128, 1, 32, 4000, TILED),     # one block per query: always
    (F32, 64, 1, 64, 4, TILED),
])
def test_filled_groups_keep_the_batch_kernels(route, dtype, dim, nq, lq, nb, kernel):
    assert route(dtype, dim, nq, lq, nb) == kernel


def test_rows_on_other_addresses(route):
    # not on 16 bytes: the documents are copied, and count as a few slots more
    assert route(BF16, 256, 2, 32, 1000, d=(1 << 30) + 2) == PAIR
    assert route(BF16, 256, 4, 32, 1000, d=(1 << 30) + 2) == KLOOP_WS
    assert route(F32, 128, 1, 32, 4000, q=(1 << 20) + 4) == PAIR
    assert route(F32, 32, 8, 32, 4000, d=(1 << 30) + 4) == PAIR  # too narrow for the K-loop


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
def test_longest_queries(route, dtype):
    assert route(dtype, 64, 40, 512, 1000) == TILED
    assert route(dtype, 64, 40, 513, 1000) == PAIR
    assert route(dtype, 768, 40, 257, 1000) == PAIR
