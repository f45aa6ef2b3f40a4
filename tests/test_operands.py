"""Alias check of plan operands on CPU tensors: byte windows of one buffer, empty tensors, in-place views.
Launch set-up on a torch that lacks the internal readings of the current stream and device."""

import importlib.util
from types import SimpleNamespace

import pytest
import torch

from venturi_amd import operands
from venturi_amd.operands import admit, disjoint


@pytest.mark.parametrize("a,b", [((0, 4), (4, 8)), ((0, 5), (4, 8)), ((4, 8), (0, 4)), ((4, 8), (0, 5)), ((2, 3), (0, 8)),
                                 ((3, 3), (0, 8)), ((0, 8), (3, 3)), ((0, 0), (0, 8)), ((2, 6), (2, 6))])
def test_disjoint_is_the_byte_windows_intersection(a, b):
    buffer = torch.zeros(8, dtype=torch.float16)
    out, operand = buffer[slice(*a)], buffer[slice(*b)]
    first, other = out.data_ptr(), operand.data_ptr()
    shared = first < other + 2 * operand.numel() and other < first + 2 * out.numel()
    for inplace in (False, True):
        if shared and not (inplace and a == b):
            with pytest.raises(ValueError, match="must not alias"):
                disjoint(out, (torch.zeros(3), operand), allow_inplace=inplace)
        else:
            disjoint(out, (torch.zeros(3), operand), allow_inplace=inplace)


@pytest.mark.parametrize("shape,dtype", [((2, 3), torch.float32), ((3, 2), torch.float16), ((6,), torch.float16)])
def test_admit_refuses_other_shapes_and_types(shape, dtype):
    where = torch.device("cpu")
    for sizes in ((2, 3), [2, 3], torch.Size((2, 3))):
        admit(torch.zeros(2, 3, dtype=torch.float16), sizes, torch.float16, where, "x")
    with pytest.raises(ValueError, match="x requires shape"):
        admit(torch.zeros(shape, dtype=dtype), (2, 3), torch.float16, where, "x")


def test_launch_setup_without_torch_internals(monkeypatch):
    for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        monkeypatch.delattr(torch._C, name, raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(cuda_stream=(7, device.index)))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    entered = []
    monkeypatch.setattr(torch.cuda, "device", lambda device: entered.append(device.index))
    spec = importlib.util.spec_from_file_location("operands_without_internals", operands.__file__)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    assert module.stream_of(torch.device("cuda", 3)) == (7, 3)
    with module.on_device(torch.device("cuda", 1)):
        assert entered == []
    module.on_device(torch.device("cuda", 0))
    assert entered == [0]
