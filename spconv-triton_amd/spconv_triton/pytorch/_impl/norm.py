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
# a subclass's operations are its own, and its memory may be none (its pointer null)
_TENSORS = (torch.Tensor, nn.Parameter)
_NAMES = frozenset(("running_mean", "running_var", "weight", "bias"))


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
    """(running mean, running variance, weight, bias) that the module's forward reads; None
    where one is not the parameter or buffer of that name (an instance attribute in its place).
    (Four reads through the module's attributes took 2 us a layer.)"""
    if not _NAMES.isdisjoint(mod.__dict__):
        return None
    params, buffers = mod._parameters, mod._buffers
    try:
        return (buffers["running_mean"], buffers["running_var"], params["weight"],
                params["bias"])
    except KeyError:
        return None


def fusable_bn(mod: nn.Module, x: torch.Tensor):
    """The statistics of ``mod`` where it is a plain eval BatchNorm1d over the rows of ``x`` that
    torch would compute from them, in types this kernel has; otherwise None."""
    if not (type(mod) is nn.BatchNorm1d and nn.BatchNorm1d.forward is _BN_FORWARD
            and not mod.training and _plain(mod)):
        return None
    if not (type(x) is torch.Tensor and x.is_cuda and x.dim() == 2 and x.is_contiguous()
            and x.dtype in _FLOATS and 0 < x.shape[1] < 65536):
        return None
    stats = _statistics(mod)
    return stats if _fusable_statistics(stats, x.dtype, x.get_device(), x.shape[1]) else None


def _fusable_statistics(stats, dtype, dev: int, width: int) -> bool:
    if stats is None or stats[0] is None or stats[1] is None:
        return False
    want = stats[0].dtype
    if want is not dtype and want is not torch.float32:
        return False
    for t in stats:
        if t is not None and not (type(t) in _TENSORS and t.dtype is want and t.get_device() == dev
                                  and t.dim() == 1 and t.numel() == width and t.is_contiguous()):
            return False
    return True


def batchnorm_eval(mod: nn.Module, x: torch.Tensor, relu: bool, stats=None) -> torch.Tensor:
    """stats: what ``fusable_bn`` returned for ``mod``."""
    out = torch.empty_like(x)
    mean, var, weight, bias = _statistics(mod) if stats is None else stats
    _lib.check(_lib.lib().sp_batchnorm_eval(
        _lib.ptr(x), _lib.dtype_code(x.dtype), x.shape[0], x.shape[1], _lib.ptr(mean),
        _lib.ptr(var), _lib.ptr(weight), _lib.ptr(bias), _lib.dtype_code(mean.dtype),
        float(mod.eps), int(relu), _lib.ptr(out), _lib.stream_of(x.device)), "sp_batchnorm_eval")
    return out
