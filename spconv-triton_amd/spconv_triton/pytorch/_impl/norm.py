"""Eval-mode BatchNorm1d (+ ReLU) of a feature tensor in one launch.

``SparseSequential`` hands the plain ``nn.BatchNorm1d`` (and the ``nn.ReLU``
after it) of an inference pass here (``sp_batchnorm_eval``).  ``fusable_bn`` and
``fusable_relu`` accept only modules whose call does nothing else: no
subclass (of module or tensors), hook, replaced ``forward``, training mode,
gradient, tracing or transform; everything else runs the modules themselves.
"""

from __future__ import annotations

import torch
from torch import nn
from torch.nn.modules import module as _module

from . import _lib

_BN_FORWARD = nn.BatchNorm1d.forward
_RELU_FORWARD = nn.ReLU.forward
_CALL = nn.Module.__call__
_FLOATS = (torch.float16, torch.bfloat16, torch.float32)
_TENSORS = (torch.Tensor, nn.Parameter)


def _plain(mod: nn.Module) -> bool:
    """Calling ``mod`` runs its class's forward and nothing else."""
    return not (mod._forward_hooks or mod._forward_pre_hooks or mod._backward_hooks
                or mod._backward_pre_hooks or mod._compiled_call_impl is not None
                or "forward" in mod.__dict__)


def passes_unobserved() -> bool:
    """No gradient, global hook, mode, trace or transform could see a module or
    tensor operation of this pass."""
    if torch.compiler.is_compiling():  # (first: Dynamo cannot trace the questions below)
        return False
    return not (torch.is_grad_enabled() or _module._global_forward_hooks
                or _module._global_forward_pre_hooks or _module._global_backward_hooks
                or _module._global_backward_pre_hooks
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0
                or torch.jit.is_tracing()
                or nn.Module.__call__ is not _CALL)


def fusable_relu(mod: nn.Module) -> bool:
    return type(mod) is nn.ReLU and nn.ReLU.forward is _RELU_FORWARD and _plain(mod)


def _statistics(mod: nn.BatchNorm1d):
    """What the module's forward reads, as it reads it (also where an instance attribute
    has taken a parameter's place)."""
    return mod.running_mean, mod.running_var, mod.weight, mod.bias


def _plain_tensor(t) -> bool:
    """The values of ``t`` are its memory's: no subclass, whose operations are its own and whose
    memory may be none, no lazy negation or zeros."""
    return type(t) in _TENSORS and not t.is_neg() and not t._is_zerotensor()


def fusable_bn(mod: nn.Module, x: torch.Tensor) -> bool:
    """``mod`` is a plain eval BatchNorm1d over the rows of ``x`` that torch would
    compute from its running statistics, in types this kernel has."""
    if not (type(mod) is nn.BatchNorm1d and nn.BatchNorm1d.forward is _BN_FORWARD
            and not mod.training and _plain(mod)):
        return False
    if not (type(x) is torch.Tensor and x.is_cuda and x.dim() == 2 and x.is_contiguous()
            and x.dtype in _FLOATS and 0 < x.shape[1] < 65536 and _plain_tensor(x)):
        return False
    return _fusable_statistics(_statistics(mod), x.dtype, x.device, x.shape[1])


def _fusable_statistics(stats, dtype, dev, width: int) -> bool:
    mean, var, weight, bias = stats
    if mean is None or var is None:
        return False
    want = mean.dtype
    if want is not dtype and want is not torch.float32:
        return False
    for t in stats:
        if t is not None and not (_plain_tensor(t) and t.dtype is want and t.device == dev
                                  and t.dim() == 1 and t.shape[0] == width
                                  and t.is_contiguous()):
            return False
    return True


def batchnorm_eval(mod: nn.Module, x: torch.Tensor, relu: bool) -> torch.Tensor:
    out = torch.empty_like(x)
    mean, var, weight, bias = _statistics(mod)
    _lib.check(_lib.lib().sp_batchnorm_eval(
        _lib.ptr(x), _lib.dtype_code(x.dtype), x.shape[0], x.shape[1], _lib.ptr(mean),
        _lib.ptr(var), _lib.ptr(weight), _lib.ptr(bias), _lib.dtype_code(mean.dtype),
        float(mod.eps), int(relu), _lib.ptr(out), _lib.stream_of(x.device)), "sp_batchnorm_eval")
    return out
