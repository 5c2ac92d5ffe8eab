"""Where the two gradients share a launch (CPU only: the host's rules).  Sharing
saves a launch, and loses where it takes CUs or waves from the longer kernel."""

from __future__ import annotations

import ctypes
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "maxsim_amd" / "libmaxsim_amd.so"
F32, F16, BF16 = 0, 1, 2
I64 = ctypes.c_int64


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(LIB))


@pytest.mark.parametrize("dtype,vec,bucket,rows,nb,dim,one", [
    (F32, 1, 1, 256, 64, 64, 1),      # 15 us in one launch, 20 in two
    (F32, 1, 1, 256, 128, 64, 1),
    (F32, 1, 1, 256, 300, 64, 0),     # 92, 80
    (F32, 1, 1, 256, 1000, 64, 0),    # 294, 258
    (F32, 1, 1, 2048, 300, 64, 1),    # 96, 101
    (F32, 1, 1, 256, 700, 128, 1),
    (F32, 1, 1, 256, 2000, 128, 0),   # 727, 559
    (F32, 1, 0, 256, 2000, 256, 0),   # 762, 680
    (F32, 1, 0, 256, 700, 256, 1),    # 193, 214
    (F32, 0, 0, 256, 2000, 300, 1),   # 1223, 1744
    (BF16, 1, 1, 256, 2000, 128, 1),  # 273, 322
    (F16, 1, 1, 256, 2000, 64, 1),
])
def test_contrastive_gradients(lib, dtype, vec, bucket, rows, nb, dim, one):
    fn = lib.maxsim_internal_contrastive_grads_one_launch
    fn.argtypes = [ctypes.c_int] * 3 + [I64] * 3
    assert fn(dtype, vec, bucket, rows, nb, dim) == one
