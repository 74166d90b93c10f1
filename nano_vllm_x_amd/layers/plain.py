"""Whether what modules compute may be computed without calling them, and what torch's operators compute without these."""
from __future__ import annotations

import torch
from torch import nn
from torch.utils._device import DeviceContext

_CALL = nn.Module.__call__
_TENSORS = (nn.Parameter, torch.Tensor)
_FORWARD = {nn.Linear: nn.Linear.forward}


def bypassable(cls):
    """Decorator of module classes that a step may pass by: remembers forward as it is written here."""
    _FORWARD[cls] = cls.forward
    return cls


def untouched(m, cls) -> bool:
    """Whether calling module `m` runs the forward that its class `cls` has, and nothing else: another class (a replaced, wrapped, quantised or
    parametrised module), a forward of the instance's own, and hooks all want the call.  (Looked up where nn.Module keeps them: a step asks this of
    every module.)  as_written says the same of the class."""
    if type(m) is not cls:      # (m.__class__ is what a proxy says of the module inside)
        return False
    d = m.__dict__
    return not d["_forward_hooks"] and not d["_forward_pre_hooks"] and "forward" not in d and "_compiled_call_impl" not in d


def as_written(*classes) -> bool:
    """Whether the classes' forwards are those that `bypassable` saw: none patched since."""
    return all(cls.forward is _FORWARD[cls] for cls in classes)


def weight_of(m):
    """The weight of a module without a bias, a plain tensor; else None (tensors of another class have operators of their own)."""
    p = m.__dict__["_parameters"]
    w = p.get("weight")
    return w if type(w) in _TENSORS and p.get("bias") is None else None


def calls_are_plain() -> bool:
    """Whether nothing stands between a call of a module and its forward, or of an operator and its kernel: no global hook or patched call, no
    autocast, function or dispatch mode (a default device is none of these), function transform, forward-mode level or tracer."""
    m = torch.nn.modules.module
    if m._global_forward_hooks or m._global_forward_pre_hooks or nn.Module.__call__ is not _CALL:
        return False
    return operators_are_plain()


def operators_are_plain() -> bool:
    c = torch._C
    modes = c._len_torch_function_stack()
    if modes and not all(type(c._get_function_stack_at(i)) is DeviceContext for i in range(modes)):
        return False
    return not (torch.is_autocast_enabled("cuda") or c._len_torch_dispatch_stack() or c._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0 or c._get_tracing_state() is not None or torch.compiler.is_compiling())
