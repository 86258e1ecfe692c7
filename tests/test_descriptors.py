"""Argument descriptors: absent slots equal those of zero-size tensors, and
every rank and type of tensor is described field by field."""

from __future__ import annotations

import pytest
import torch

from beamz_amd import native


def _fields(b):
    return (b.data, b.rank, b.element_type, tuple(b.dims))


@pytest.mark.parametrize("shape,dtype", [((0,), torch.float32), ((0, 1, 1, 1), torch.float32),
                                         ((0, 1), torch.float32), ((0, 3), torch.int32)])
def test_absent_matches_empty_tensor(shape, dtype):
    assert _fields(native.buffer(native.Absent(shape, dtype))) == \
        _fields(native.buffer(torch.zeros(shape, dtype=dtype)))


@pytest.mark.parametrize("shape", [(), (5,), (2, 3), (4, 1, 2), (1, 2, 3, 4)])
@pytest.mark.parametrize("dtype,code", [(torch.float32, native.F32), (torch.float64, native.F64)])
def test_tensor_fields(shape, dtype, code):
    t = torch.ones(shape, dtype=dtype)
    arr = native.buffers([None, t])
    assert _fields(arr[0]) == (None, 1, native.F32, (0, 0, 0, 0))
    assert _fields(arr[1]) == (t.data_ptr(), len(shape), code, (*shape, 0, 0, 0, 0)[:4])


def test_refusals():
    with pytest.raises(native.HipLaunchError):
        native.buffer(torch.ones(3, 4).t())
    with pytest.raises(native.HipLaunchError):
        native.buffer(torch.ones(1, 1, 1, 1, 1))
