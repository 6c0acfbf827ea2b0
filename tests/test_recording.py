"""When a kernel may stand in for PyTorch ops that something else is watching (smlm_hip.recording)."""
import pytest
from torch import nn
from torch.nn.modules import module as nn_module

from smlm_hip.recording import unhooked


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
