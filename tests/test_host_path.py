"""Shortcuts of the operators' host path against the general calls they stand for."""
import pytest
import torch

from apr_models.unet import unet_model
from pyapr.aprnet import _ops


def test_submodules_are_those_of_modules():
    shared = torch.nn.ReLU()
    net = torch.nn.Sequential(torch.nn.Linear(2, 2), shared, torch.nn.ModuleList([torch.nn.Sequential(shared, torch.nn.Identity())]))
    net.register_module("nothing", None)
    mine = list(unet_model._submodules(net))
    assert len(mine) == len(set(mine)) and set(mine) == set(net.modules()) - {net}


def test_flags_of_instances_and_classes():
    class Off(torch.nn.Identity):
        increment_level_deltas = False
    m = torch.nn.Identity()
    assert unet_model._flag(m, "increment_level_deltas") is True and unet_model._flag(Off(), "increment_level_deltas") is False
    m.increment_level_deltas = False
    assert unet_model._flag(m, "increment_level_deltas") is False


@pytest.mark.parametrize("t", [torch.zeros(3, 4, 5), torch.zeros(6, 4, 5, dtype=torch.bfloat16)[::2], torch.zeros(3, 4, 5).transpose(0, 2)])
def test_address_of_a_batch_item(t):
    for b in range(t.shape[0]):
        assert _ops._at(t, b).value == t[b].data_ptr()
    with pytest.raises(IndexError):
        _ops._at(t, t.shape[0])


@pytest.mark.gpu
def test_stream_and_device_of_a_call():
    s = torch.cuda.Stream()
    with torch.cuda.stream(s), _ops._on(torch.device("cuda", torch.cuda.current_device())):
        assert _ops._stream().value == s.cuda_stream
    assert (_ops._stream().value or 0) == torch.cuda.current_stream().cuda_stream
    assert isinstance(_ops._on("cuda"), torch.cuda.device)          # anything else goes the general way
