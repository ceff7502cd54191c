"""Eval BatchNorm1d (+ ReLU) inside SparseSequential: the one-launch kernel against
fp64 and against torch's modules, and the modules it must leave to torch."""

import numpy as np
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
UNIT = {F16: 2.0 ** -11, BF16: 2.0 ** -8, F32: 2.0 ** -24}


def _tensor(feats):
    import spconv_triton.pytorch as spconv

    n = feats.shape[0]
    idx = np.stack([np.zeros(n), np.arange(n) // 64 // 64, np.arange(n) // 64 % 64,
                    np.arange(n) % 64], 1).astype(np.int32)
    return spconv.SparseConvTensor(feats, torch.from_numpy(idx).to(DEV), [64, 64, 64], 1)


def _bn(C, dtype, affine=True, seed=0):
    g = torch.Generator().manual_seed(seed)
    bn = nn.BatchNorm1d(C, affine=affine)
    with torch.no_grad():
        bn.running_mean.copy_(torch.randn(C, generator=g))
        bn.running_var.copy_(torch.rand(C, generator=g) * 2 + 0.01)
        if affine:
            bn.weight.copy_(torch.randn(C, generator=g))
            bn.bias.copy_(torch.randn(C, generator=g))
    return bn.to(DEV).to(dtype).eval()


@pytest.mark.parametrize("rows,C,dtype,pdtype,affine,relu", [
    (1, 16, F16, F16, True, True), (4097, 32, F16, F16, True, True),
    (255, 2048, F16, F32, True, False), (255, 2056, F16, F16, True, True),  # past 256 pieces
    (1000, 20, F16, F16, True, True), (513, 3, F16, F16, True, False),  # no whole vectors
    (777, 48, BF16, BF16, True, True), (777, 64, BF16, F32, False, True),
    (4097, 64, F32, F32, True, True), (33, 5, F32, F32, False, False)])
def test_batchnorm_eval_matches_fp64(rows, C, dtype, pdtype, affine, relu):
    """|error| <= 1 rounding of the result's type + 8 fp32 roundings of the terms."""
    import spconv_triton.pytorch as spconv

    torch.manual_seed(rows + C)
    x = torch.randn(rows, C, device=DEV).to(dtype)
    bn = _bn(C, pdtype, affine)
    net = spconv.SparseSequential(bn, *([nn.ReLU()] if relu else []))
    with torch.no_grad():
        y = net(_tensor(x)).features
        t = bn(x)
        t = torch.relu(t) if relu else t
    m, v = bn.running_mean.double(), bn.running_var.double()
    w = bn.weight.double() if affine else torch.ones_like(m)
    b = bn.bias.double() if affine else torch.zeros_like(m)
    scale = w / torch.sqrt(v + bn.eps)
    ref = (x.double() - m) * scale + b
    mag = (x.double().abs() + m.abs()) * scale.abs() + b.abs()
    ref = ref.clamp(min=0) if relu else ref
    bound = UNIT[dtype] * ref.abs() + 8 * 2.0 ** -24 * mag + (2.0 ** -25 if dtype is F16 else 0)
    assert y.dtype == dtype and ((y.double() - ref).abs() <= bound).all()
    assert ((y.double() - t.double()).abs() <= 2 * bound).all()


def test_batchnorm_special_values():
    import spconv_triton.pytorch as spconv

    x = torch.randn(64, 16, device=DEV).half()
    x[3, 2], x[4, 5], x[5, 7] = float("nan"), float("inf"), -float("inf")
    bn = _bn(16, F16)
    with torch.no_grad():
        y = spconv.SparseSequential(bn, nn.ReLU())(_tensor(x)).features
        t = torch.relu(bn(x))
    assert torch.equal(torch.isnan(y), torch.isnan(t)) and torch.isnan(y[3, 2])
    assert torch.equal(torch.isinf(y), torch.isinf(t))


@pytest.mark.parametrize("rows,C,dtype,pdtype,affine", [
    (1, 16, F16, F16, True), (20000, 64, F16, F16, True), (3001, 33, F16, F32, True),
    (3000, 2056, F16, F16, True), (5000, 128, F16, F16, False), (9000, 48, BF16, BF16, True),
    (2000, 5, BF16, F32, False), (9000, 64, F32, F32, True), (700, 300, F32, F32, False),
    (129, 1030, F32, F32, True)])
def test_batchnorm_eval_is_torch_bit_for_bit(rows, C, dtype, pdtype, affine):
    """The steps and their order are the module's, so a network's values do not depend on
    whether its BatchNorm and ReLU are fused."""
    import spconv_triton.pytorch as spconv

    torch.manual_seed(rows + C)
    x = (torch.randn(rows, C, device=DEV) * 2).to(dtype)
    bn = _bn(C, pdtype, affine, seed=C)
    x[0] = bn.running_mean.to(dtype)
    bits = torch.int32 if dtype is F32 else torch.int16
    with torch.no_grad():
        t = bn(x)
        for net, ref in ((spconv.SparseSequential(bn), t),
                         (spconv.SparseSequential(bn, nn.ReLU()), torch.relu(t))):
            y = net(_tensor(x)).features
            assert torch.equal(y.view(bits), ref.view(bits))


class _MyBN(nn.BatchNorm1d):
    def forward(self, x):
        return super().forward(x) + 1


def test_observed_modules_run_themselves(monkeypatch):
    """Hooks, subclasses, replaced forwards, training mode and gradients keep torch's modules."""
    import spconv_triton.pytorch as spconv
    from spconv_triton.pytorch._impl import norm

    calls = []
    real = norm.batchnorm_eval
    monkeypatch.setattr(norm, "batchnorm_eval",
                        lambda *a: (calls.append(1), real(*a))[1])
    x = torch.randn(100, 16, device=DEV)
    bn, relu = _bn(16, F32), nn.ReLU()
    net = spconv.SparseSequential(bn, relu)
    with torch.no_grad():
        net(_tensor(x))
        assert len(calls) == 1
        for mod in (bn, relu):  # a hook on either is called
            seen = []
            h = mod.register_forward_hook(lambda m, i, o: seen.append(o))
            y = net(_tensor(x)).features
            h.remove()
            assert len(seen) == 1 and torch.equal(seen[0].clamp(min=0), y)
        assert len(calls) == 2  # the ReLU's hook left the BatchNorm fusable
        relu.forward = lambda v: v * 2
        assert torch.equal(net(_tensor(x)).features, real(bn, x, False) * 2)
        del relu.forward
        my = _MyBN(16).to(DEV).eval()
        my.load_state_dict(bn.state_dict())
        n = len(calls)
        torch.testing.assert_close(spconv.SparseSequential(my)(_tensor(x)).features, bn(x) + 1)
        spconv.SparseSequential(bn.train())(_tensor(x))
        bn.eval()
        assert len(calls) == n
    y = net(_tensor(x.clone().requires_grad_(True))).features
    assert y.requires_grad and len(calls) == n


class _Doubled(torch.Tensor):
    """A tensor without memory of its own whose value is twice the one it holds."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype,
                                                   device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        args = [a.inner * 2 if isinstance(a, cls) else a for a in args]
        return func(*args, **(kwargs or {}))


def test_other_parameters_than_plain_tensors():
    """A wrapper-subclass weight, or an attribute in the parameter's place, counts."""
    import spconv_triton.pytorch as spconv

    x = torch.randn(100, 16, device=DEV)
    bn = _bn(16, F32)
    weight = bn.weight.detach().clone()
    net = spconv.SparseSequential(bn, nn.ReLU())
    with torch.no_grad():
        bn.weight.mul_(2)
        want = torch.relu(bn(x))
        bn._parameters["weight"] = _Doubled(weight)
        assert torch.equal(net(_tensor(x)).features, want)
        del bn.weight
        bn.weight = weight * 2
        assert torch.equal(net(_tensor(x)).features, want)
