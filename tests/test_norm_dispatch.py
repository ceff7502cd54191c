"""Which BatchNorm1d and ReLU modules SparseSequential may run as one launch: the parts of the
choice that need no GPU."""

import pytest
import torch
from torch import nn

CPU = -1  # torch's device index of host tensors


def _tensor(feats):
    import spconv_triton.pytorch as spconv

    n = feats.shape[0]
    idx = torch.stack([torch.zeros(n), torch.arange(n), torch.arange(n), torch.arange(n)], 1).int()
    return spconv.SparseConvTensor(feats, idx, [n, n, n], 1)


@pytest.mark.parametrize("grad", [False, True])
def test_sequential_compiles_to_one_graph(grad):
    import spconv_triton.pytorch as spconv

    net = spconv.SparseSequential(nn.BatchNorm1d(4), nn.ReLU()).eval()
    net[0].running_mean.copy_(torch.tensor([0.5, -1.0, 2.0, 0.0]))
    x = torch.randn(6, 4, generator=torch.Generator().manual_seed(0))

    def run(feats):
        return net(_tensor(feats)).features

    with torch.set_grad_enabled(grad):
        y = torch.compile(run, fullgraph=True, backend="eager")(x)
        assert torch.equal(y, torch.relu(net[0](x)))


class _Wrapper(torch.Tensor):
    """A tensor that holds another one and has no memory of its own (quantised and
    distributed parameters are such)."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype,
                                                   device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        def open_(v):
            return v.inner * 2 if isinstance(v, cls) else v
        args = [open_(a) for a in args]
        return func(*args, **{k: open_(v) for k, v in (kwargs or {}).items()})


class _Observed(torch.Tensor):
    """A subclass whose operations are its own."""


def _statistics(**changed):
    from spconv_triton.pytorch._impl import norm

    bn = nn.BatchNorm1d(4).eval()
    for name, t in changed.items():
        if name in bn._buffers:
            bn._buffers[name] = t
        else:
            bn._parameters[name] = t
    return norm._statistics(bn)


@pytest.mark.parametrize("name", ["running_mean", "running_var", "weight", "bias"])
@pytest.mark.parametrize("make,ok", [
    (lambda t: t, True), (nn.Parameter, True), (lambda t: _Wrapper(t), False),
    (lambda t: t.as_subclass(_Observed), False), (lambda t: t.double(), False),
    (lambda t: torch.ones(8)[::2], False), (lambda t: torch.ones(5), False)])
def test_only_plain_statistics_are_fused(name, make, ok):
    """A wrapper subclass has no memory (its pointer would read as "no weight")."""
    from spconv_triton.pytorch._impl import norm

    stats = _statistics(**{name: make(torch.ones(4))})
    assert norm._fusable_statistics(stats, torch.float32, CPU, 4) == ok


def test_an_attribute_in_a_parameters_place_is_not_fused():
    """(Its value would read as "no weight".)  Nor is a module that has lost a parameter."""
    from spconv_triton.pytorch._impl import norm

    for replace in (True, False):
        bn = nn.BatchNorm1d(4).eval()
        del bn.weight
        if replace:
            bn.weight = torch.full((4,), 3.0)
        assert not norm._fusable_statistics(norm._statistics(bn), torch.float32, CPU, 4)


def test_no_affine_and_half_types():
    from spconv_triton.pytorch._impl import norm

    plain = norm._statistics(nn.BatchNorm1d(4, affine=False))
    assert plain[2] is None and norm._fusable_statistics(plain, torch.float16, CPU, 4)
    assert not norm._fusable_statistics(
        norm._statistics(nn.BatchNorm1d(4, track_running_stats=False)), torch.float32, CPU, 4)
    assert not norm._fusable_statistics(
        norm._statistics(nn.BatchNorm1d(4).half()), torch.bfloat16, CPU, 4)
