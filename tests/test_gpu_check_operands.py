"""The layout-check operators called directly: arrays on other devices and
tensors that are no check's result are refused before anything is launched or
waited for."""

from __future__ import annotations

import pytest
import torch

from maxsim_amd._ops import ops

from ._helpers import DEVICE

pytestmark = pytest.mark.gpu


def _i32(*values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def test_host_array_beside_a_device_one_is_refused():
    off, ids, lens = _i32(0, 3, 5), _i32(0, 1), _i32(2, 2)
    calls = [
        (ops.maxsim_check_padded, [lens, lens], (4, 4)),
        (ops.maxsim_check_packed, [off, off, ids, ids], (5, 5)),
        (lambda o, t: ops.maxsim_check_contrastive(o, 5, t), [off, ids], ()),
    ]
    for fn, arrays, rest in calls:
        status = fn(*arrays, *rest)
        assert ops.maxsim_check_wait(status, off) >= 0
        for at in range(len(arrays)):
            moved = list(arrays)
            moved[at] = moved[at].cpu()
            with pytest.raises(RuntimeError, match="one HIP"):
                fn(*moved, *rest)


def test_wait_refuses_tensors_that_are_no_check():
    off = _i32(0, 3, 5)
    status = ops.maxsim_check_contrastive(off, 5, None)
    assert ops.maxsim_check_wait(status, off) == 3
    done = torch.ones_like(status)  # looks finished, its stream is not one
    for other in (status.clone(), status[:-1], status.to(torch.int32), status.to(DEVICE), done,
                  torch.zeros(1, dtype=torch.int64)):
        with pytest.raises(RuntimeError, match="layout check"):
            ops.maxsim_check_wait(other, off)
