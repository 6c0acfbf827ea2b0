"""When a kernel may stand in for a sequence of PyTorch ops that other machinery could be watching."""
import torch
from torch.autograd import forward_ad
from torch.nn.modules import module as nn_module
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext


def _function_mode():
    """Whether a torch function mode is active that sees more than factory calls (a default device does not)."""
    return (torch._C._is_torch_function_mode_enabled()
            and any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()))


def ordinary(*tensors):
    """Whether nothing but eager execution and reverse-mode recording sees these tensors: plain tensors, and no
    compilation, tracing, function transform (vmap, grad, jvp), forward-mode level, function mode or dispatch mode is
    active.  Else the PyTorch ops run, which all of these follow."""
    return (all(t is None or type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors)
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and not torch._C._are_functorch_transforms_active() and forward_ad._current_level < 0
            and torch._C._len_torch_dispatch_stack() == 0 and not _function_mode())


def unhooked(*modules):
    """Whether these modules' calls do nothing but their class's forward (no hooks of their own, none on all modules, no
    forward put on the module), so that a kernel may read their weights."""
    if (nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks or nn_module._global_backward_hooks
            or nn_module._global_backward_pre_hooks):
        return False
    for m in modules:
        own = m.__dict__
        if (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or own["_backward_pre_hooks"]
                or "forward" in own):
            return False
    return True


def records(*tensors):
    """Whether autograd records an op on these tensors."""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)
