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
    (F32, 1, 0, 64, 2000, 96, 1),     # 381, 443
    (F32, 0, 0, 256, 2000, 300, 1),   # 1223, 1744
    (BF16, 1, 1, 256, 2000, 128, 1),  # 273, 322
    (F16, 1, 1, 256, 2000, 64, 1),
])
def test_contrastive_gradients(lib, dtype, vec, bucket, rows, nb, dim, one):
    fn = lib.maxsim_internal_contrastive_grads_one_launch
    fn.argtypes = [ctypes.c_int] * 3 + [I64] * 3
    assert fn(dtype, vec, bucket, rows, nb, dim) == one


@pytest.mark.parametrize("out16,whole_rows,rows,dim,one", [
    (1, 0, 4096 * 300, 768, 0),   # 512 us in one launch, 454 in two
    (1, 0, 4096 * 300, 100, 0),   # 112, 98
    (1, 0, 1024 * 300, 100, 1),   # 37, 37
    (1, 0, 64 * 300, 768, 1),     # 27, 33
    (1, 1, 16384 * 300, 256, 1),  # 446, 521
    (0, 1, 4096 * 300, 256, 0),   # 284, 250
    (0, 1, 3200 * 100, 128, 1),   # 39, 44
    (0, 0, 1024 * 600, 768, 1),   # 399, 454
])
def test_padded_gradients(lib, out16, whole_rows, rows, dim, one):
    fn = lib.maxsim_internal_padded_grads_one_launch
    fn.argtypes = [ctypes.c_int, ctypes.c_int, I64]
    assert fn(out16, whole_rows, rows * dim * (2 if out16 else 4)) == one
