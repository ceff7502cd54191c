"""The narrow GEMM (outputs of at most 32 columns without a plan): bit-identical to the
planned kernels over row widths on both sides of its instances (whole 16-byte pieces,
8-byte halves, single elements; one or two K-steps; several chunks), tile edges, windows
of several offset groups and tables without pairs."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("C,K", [(3, 32), (4, 16), (8, 8), (12, 20), (16, 32), (17, 31), (20, 5),
                                 (32, 32), (36, 24), (64, 1), (96, 32)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_narrow_equals_planned(C, K, dtype, monkeypatch):
    from spconv_triton.pytorch._impl import gemm

    monkeypatch.setattr(gemm, "ROW_ORDER", "natural")
    rng = np.random.default_rng(C * 100 + K)
    for M, kv, density in ((1, 27, 0.5), (255, 27, 0.1), (257, 3, 0.9), (700, 1, 1.0),
                           (1000, 64, 0.02), (64, 9, 0.0)):
        n_src = M + 3
        t = rng.integers(0, n_src, size=(kv, M)).astype(np.int32)
        t[rng.random((kv, M)) >= density] = -1
        tab = torch.from_numpy(t).to(DEV)
        g = torch.Generator(device=DEV)
        g.manual_seed(M)
        x = torch.randn(n_src, C, generator=g, device=DEV).to(dtype)
        w = torch.randn(K, kv, C, generator=g, device=DEV).to(dtype)
        b = torch.randn(K, generator=g, device=DEV).to(dtype)
        for out_dtype in (dtype, torch.float32):
            monkeypatch.setattr(gemm, "USE_GATHER_PLAN", False)
            got = gemm.conv_forward(x, w, tab, M, bias=b, out_dtype=out_dtype)
            monkeypatch.setattr(gemm, "USE_GATHER_PLAN", True)
            want = gemm.conv_forward(x, w, tab.clone(), M, bias=b, out_dtype=out_dtype)
            assert torch.equal(got, want), (M, kv, out_dtype)


def test_narrow_large_window_matches_fp64():
    """kv > 64: three groups of offsets (the planned kernels do not take them)."""
    from spconv_triton.pytorch._impl.gemm import conv_forward

    rng = np.random.default_rng(0)
    kv, M, C, K = 150, 300, 24, 20
    t = rng.integers(0, M, size=(kv, M)).astype(np.int32)
    t[rng.random((kv, M)) >= 0.1] = -1
    tab = torch.from_numpy(t).to(DEV)
    x = torch.randn(M, C, device=DEV)
    w = torch.randn(K, kv, C, device=DEV)
    y = conv_forward(x, w, tab, M)
    ref = torch.zeros(M, K, dtype=torch.float64, device=DEV)
    mag = torch.zeros_like(ref)
    for k in range(kv):
        o = torch.nonzero(tab[k] >= 0).view(-1)
        xi = x[tab[k][o].long()].double()
        ref[o] += xi @ w[:, k].double().T
        mag[o] += xi.abs() @ w[:, k].double().abs().T
    # at most 150 * 24 fp32 sums of exact-to-rounding products
    assert ((y.double() - ref).abs() <= 2.0 ** -24 * 200 * mag + 1e-30).all()


@pytest.mark.parametrize("C,K,dtype", [(64, 32, torch.float32), (16, 32, torch.float16),
                                       (4, 16, torch.bfloat16)])
def test_a_table_in_mask_order_keeps_its_plan(C, K, dtype, monkeypatch):
    """A narrow layer on a table whose rows are taken in mask order runs the planned kernel: the
    narrow one takes natural rows only.  The result is that of the narrow kernel."""
    from spconv_triton.pytorch._impl import gemm

    rng = np.random.default_rng(C)
    kv, M = 27, 1500
    t = rng.integers(0, M, size=(kv, M)).astype(np.int32)
    t[rng.random((kv, M)) >= 0.1] = -1
    x = torch.randn(M, C, device=DEV).to(dtype)
    w = torch.randn(K, kv, C, device=DEV).to(dtype)
    monkeypatch.setattr(gemm, "PLAN_MIN_WORK", M * K)
    plain = torch.from_numpy(t).to(DEV)
    monkeypatch.setattr(gemm, "ROW_ORDER", "natural")
    want = gemm.conv_forward(x, w, plain, M)
    assert not hasattr(plain, "_spconv_triton_plan")  # the narrow kernel
    ordered = torch.from_numpy(t).to(DEV)
    monkeypatch.setattr(gemm, "ROW_ORDER", "mask")
    got = gemm.conv_forward(x, w, ordered, M)
    assert ordered._spconv_triton_order[1][2] is not None
    assert torch.equal(got, want)


def test_output_types_the_narrow_kernel_does_not_write_are_planned(monkeypatch):
    from spconv_triton.pytorch._impl import gemm

    monkeypatch.setattr(gemm, "ROW_ORDER", "natural")
    monkeypatch.setattr(gemm, "PLAN_MIN_WORK", 1)
    tab = torch.arange(300, dtype=torch.int32, device=DEV).view(1, -1)
    x = torch.randn(300, 8, device=DEV).half()
    w = torch.randn(8, 1, 8, device=DEV).half()
    y = gemm.conv_forward(x, w, tab, 300, out_dtype=torch.bfloat16)
    assert hasattr(tab, "_spconv_triton_plan")
    ref = gemm.conv_forward(x, w, tab, 300, out_dtype=torch.float32)
    assert torch.equal(y, ref.bfloat16())
