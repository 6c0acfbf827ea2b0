"""When a kernel may stand in for PyTorch ops that something else is watching (smlm_hip.recording)."""
import pytest
import torch
from torch import nn
from torch.nn.modules import module as nn_module
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from smlm_hip.recording import ordinary, unhooked


def _nothing(*args, **kwargs):
    return None


@pytest.mark.parametrize("register", ["register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
                                      "register_full_backward_pre_hook"])
def test_a_module_with_a_hook_is_called(register):
    watched, plain = nn.Linear(2, 2), nn.Linear(2, 2)
    handle = getattr(watched, register)(_nothing)
    assert not unhooked(plain, watched) and unhooked(plain)
    handle.remove()
    assert unhooked(plain, watched)


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                      "register_module_full_backward_hook", "register_module_full_backward_pre_hook"])
def test_every_module_is_called_under_a_global_hook(register):
    plain = nn.Linear(2, 2)
    handle = getattr(nn_module, register)(_nothing)
    try:
        assert not unhooked(plain)
    finally:
        handle.remove()
    assert unhooked(plain)


def test_a_module_with_a_forward_of_its_own_is_called():
    watched = nn.Linear(2, 2)
    watched.forward = _nothing
    assert not unhooked(watched)
    del watched.forward
    assert unhooked(watched)


class _Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Dispatches(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode", [_Functions, _Dispatches])
def test_nothing_is_ordinary_under_a_mode(mode):
    x = torch.zeros(2)
    with mode():
        assert not ordinary(x)
        with torch.device("cpu"):
            assert not ordinary(x)
    assert ordinary(x)


def test_a_default_device_is_ordinary():
    """torch.device as a context and set_default_device are function modes that touch factory calls only."""
    x = torch.zeros(2)
    with torch.device("cpu"):
        assert ordinary(x)
    torch.set_default_device("cpu")
    try:
        assert ordinary(x)
    finally:
        torch.set_default_device(None)
    assert ordinary(x)
