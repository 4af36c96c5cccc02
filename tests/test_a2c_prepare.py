"""The native preparation of sequences leaves calls that are not plain to the
layer's Python code: under a mode the buffers that it fills need not have memory."""
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from torchproteinlibrary_amd._native_xform import ext


def test_prepare_leaves_calls_under_modes_alone():
    with FakeTensorMode():
        assert ext.Angles2Coords_prepare(["ACD", "G"], torch.empty(2, 8, 3, device="cuda")) is None
    assert ext.Angles2Coords_prepare(["ACD", "G"], torch.empty(2, 8, 3)) is None
    assert ext.Angles2Coords_prepare([], torch.empty(0, 8, 3)) is None
