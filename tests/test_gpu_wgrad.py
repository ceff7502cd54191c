"""The weight gradient's pair compaction and shares at the sizes where they can
go wrong: chunks and runs of the compaction cut short, offsets without pairs,
one offset with nearly all of them, more offsets than a workgroup looks at in
one turn, rows of no whole vector, and blocks on both sides of the reduction's
two instances."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _table(kv, n, n_in, density, seed):
    """[kv, n] gather table; density of offset k: density[k % len(density)]."""
    rng = np.random.default_rng(seed)
    t = rng.integers(0, n_in, size=(kv, n), dtype=np.int32)
    keep = rng.random((kv, n)) < np.asarray(density)[np.arange(kv) % len(density)][:, None]
    return np.where(keep, t, -1).astype(np.int32)


@pytest.mark.parametrize("kv,n,density", [
    (1, 1, [1.0]), (3, 63, [0.0, 1.0, 0.3]), (27, 1024, [0.1]), (27, 1025, [0.02, 1.0]),
    (8, 64 * 1024, [0.5]), (5, 65 * 1024 + 3, [0.001, 0.9]), (300, 700, [0.05, 0.0, 0.4])])
def test_compaction_matches_numpy(kv, n, density):
    from spconv_triton.pytorch._impl import _lib
    from spconv_triton.pytorch._impl.gemm import compacted_signal

    t = _table(kv, n, 1000, density, kv + n)
    tab = torch.from_numpy(t).to(DEV)
    in_rows, out_rows, counts = compacted_signal(tab)
    # the same lists with -1 tails and limited counts (the Native format)
    L = _lib.lib()
    pos, val = torch.empty_like(tab), torch.empty_like(tab)
    npl = torch.empty(kv, dtype=torch.int32, device=DEV)
    ws = _lib.workspace(L.sp_compact_workspace_size(kv, n), tab.device)
    _lib.check(L.sp_compact_table(_lib.ptr(tab), kv, n, _lib.ptr(pos), _lib.ptr(val), None,
                                  _lib.ptr(npl), kv // 2, _lib.ptr(ws), ws.numel(),
                                  _lib.stream_of(tab.device)), "sp_compact_table")
    pos, val, npl = pos.cpu().numpy(), val.cpu().numpy(), npl.cpu().numpy()
    in_rows, out_rows, counts = (v.cpu().numpy() for v in (in_rows, out_rows, counts))
    for k in range(kv):
        cols = np.nonzero(t[k] >= 0)[0]
        m = cols.size
        assert counts[k] == m and npl[k] == (m if k < kv // 2 else 0)
        for got_pos, got_val in ((pos[k], val[k]), (out_rows[k], in_rows[k])):
            np.testing.assert_array_equal(got_pos[:m], cols)
            np.testing.assert_array_equal(got_val[:m], t[k, cols])
        assert (pos[k, m:] == -1).all() and (val[k, m:] == -1).all()


CENTRE = [0.001] * 13 + [1.0] + [0.001] * 13  # a dense centre, as of a sparse submanifold table


@pytest.mark.parametrize("kv,n,C,K,density,dtype", [
    (27, 3000, 64, 64, [0.05], torch.float16),
    (27, 40000, 64, 64, CENTRE, torch.float16),
    (27, 40000, 160, 128, CENTRE, torch.bfloat16),
    (27, 20000, 128, 128, CENTRE, torch.float32),
    (27, 9000, 64, 128, [1.0], torch.float16),  # every entry a pair
    (300, 500, 32, 16, [0.0, 0.2], torch.float32),  # the offsets' shares in several looks
    (600, 400, 16, 16, [0.0, 0.3], torch.float16),  # more offsets than workgroups aimed at
    (64, 300, 16, 16, [0.0] * 63 + [1.0], torch.float16),  # the last of a wave's offsets
    (65, 300, 16, 16, [0.0] * 64 + [1.0], torch.float16),  # the first of the next look
    (8, 129, 256, 256, [1.0], torch.float16),  # one stage and one pair
    (27, 2000, 3, 20, [0.1], torch.float16),  # rows of no whole vector
    (9, 3000, 130, 200, [0.5], torch.float16),  # 128-wide blocks, one side in vectors
    (9, 3000, 131, 201, [0.5], torch.float32),  # and none
    (1, 1, 16, 16, [1.0], torch.float32),
    (3, 50, 16, 16, [0.0], torch.float16),  # no pairs at all
    (9, 5000, 72, 120, [0.3], torch.float32),
    (2, 700, 5, 7, [0.0, 0.5], torch.float32),  # an offset without pairs, scalar reduction
])
@pytest.mark.parametrize("tf32", [False, True])
def test_every_pair_counts_once(kv, n, C, K, density, dtype, tf32, monkeypatch):
    """Small whole numbers: every sum is exact in fp32, so the result is the fp64 one rounded, and
    a pair that is lost or counted twice shows."""
    from spconv_triton import constants
    from spconv_triton.pytorch._impl.gemm import conv_backward_weight

    if tf32 and dtype is not torch.float32:
        pytest.skip("fp32 operands only")
    monkeypatch.setattr(constants, "SPCONV_ALLOW_TF32", tf32)
    n_in = n + 17
    t = _table(kv, n, n_in, density, kv * 7 + n)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    x = torch.randint(-2, 3, (n_in, C), generator=g, device=DEV).to(dtype)
    go = torch.randint(-1, 2, (n, K), generator=g, device=DEV).to(dtype)
    tab = torch.from_numpy(t).to(DEV)
    dw = conv_backward_weight(x, go, tab, (K, kv, C))
    assert torch.equal(dw, conv_backward_weight(x, go, tab, (K, kv, C)))
    for k in range(kv):
        o = torch.nonzero(tab[k] >= 0).view(-1)
        ref = go[o].double().T @ x[tab[k][o].long()].double()
        assert torch.equal(dw[:, k], ref.to(dtype)), f"offset {k}"


@pytest.mark.parametrize("kv,n,C,K,density,dtype", [
    (27, 3000, 64, 64, [0.05], torch.float16), (27, 2000, 128, 160, [0.3], torch.bfloat16),
    (300, 500, 32, 16, [0.0, 0.2], torch.float32), (9, 2500, 72, 120, [0.3], torch.float32)])
def test_shares_match_fp64(kv, n, C, K, density, dtype):
    """|error| <= u_out |result| + pairs 2^-24 sum |x||g|: the result's own rounding and an
    offset's pairs in one chain of fp32 sums (products of 16-bit values are exact, an fp32
    product adds one rounding)."""
    from spconv_triton.pytorch._impl.gemm import conv_backward_weight

    n_in = n + 17
    t = _table(kv, n, n_in, density, kv * 7 + n)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    x = torch.randn(n_in, C, generator=g, device=DEV).to(dtype)
    go = torch.randn(n, K, generator=g, device=DEV).to(dtype)
    tab = torch.from_numpy(t).to(DEV)
    dw = conv_backward_weight(x, go, tab, (K, kv, C))
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
    for k in range(kv):
        o = torch.nonzero(tab[k] >= 0).view(-1)
        xi, gi = x[tab[k][o].long()].double(), go[o].double()
        ref, mag = gi.T @ xi, gi.abs().T @ xi.abs()
        bound = unit * ref.abs() + (o.numel() + 1) * 2.0 ** -24 * mag * (1 + unit) + 1e-30
        assert ((dw[:, k].double() - ref).abs() <= bound).all(), f"offset {k}"


def _call(x, go, tab, K, ws, dw):
    """sp_conv_wgrad with the caller's own buffers."""
    from spconv_triton.pytorch._impl import _lib
    from spconv_triton.pytorch._impl.gemm import compacted_signal

    in_rows, out_rows, counts = compacted_signal(tab)
    kv, n = tab.shape
    _lib.check(_lib.lib().sp_conv_wgrad(
        _lib.ptr(x), x.shape[0], _lib.ptr(go), n, _lib.dtype_code(x.dtype), x.shape[1], K, kv,
        _lib.ptr(in_rows), _lib.ptr(out_rows), _lib.ptr(counts), n, _lib.ptr(dw), _lib.ptr(ws),
        ws.numel(), _lib.stream_of(x.device)), "sp_conv_wgrad")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("ws_off,dw_off", [(0, 0), (4, 0), (0, 1), (12, 3), (1, 2)])
def test_buffers_at_any_address(dtype, ws_off, dw_off):
    """The workspace may start at any byte and dW at any element; nothing is written past them."""
    from spconv_triton.pytorch._impl import _lib
    from spconv_triton.pytorch._impl.gemm import conv_backward_weight

    kv, n, C, K = 5, 700, 20, 24
    tab = torch.from_numpy(_table(kv, n, n, [0.5, 0.1], 3)).to(DEV)
    g = torch.Generator(device=DEV)
    g.manual_seed(1)
    x = torch.randn(n, C, generator=g, device=DEV).to(dtype)
    go = torch.randn(n, K, generator=g, device=DEV).to(dtype)
    size = _lib.lib().sp_wgrad_workspace_size(K, kv, C, n)
    ws = torch.full((size + 64,), 0xA5, dtype=torch.uint8, device=DEV)
    out = torch.full((K * kv * C + 8,), 7.0, dtype=dtype, device=DEV)
    _call(x, go, tab, K, ws[ws_off:ws_off + size], out[dw_off:])
    want = conv_backward_weight(x, go, tab, (K, kv, C)).view(-1)
    assert torch.equal(out[dw_off:dw_off + want.numel()], want)
    assert (out[:dw_off] == 7).all() and (out[dw_off + want.numel():] == 7).all()
    assert (ws[:ws_off] == 0xA5).all() and (ws[ws_off + size:] == 0xA5).all()


def test_a_table_edited_in_place_is_compacted_again():
    from spconv_triton.pytorch._impl.gemm import compacted_signal, conv_backward_weight

    kv, n, C, K = 9, 500, 16, 16
    tab = torch.from_numpy(_table(kv, n, n, [0.4], 5)).to(DEV)
    x = torch.randn(n, C, device=DEV)
    go = torch.randn(n, K, device=DEV)
    conv_backward_weight(x, go, tab, (K, kv, C))
    assert compacted_signal(tab)[2] is compacted_signal(tab)[2]
    tab[:, ::3] = -1
    want = conv_backward_weight(x, go, tab.clone(), (K, kv, C))
    assert torch.equal(conv_backward_weight(x, go, tab, (K, kv, C)), want)


def test_weights_of_a_billion_values():
    """K * C = 2^30: entries are counted in 32 unsigned bits, their addresses in 64."""
    from spconv_triton.pytorch._impl.gemm import conv_backward_weight

    C = K = 32768
    g = torch.Generator(device=DEV)
    g.manual_seed(2)
    x = torch.randint(-2, 3, (5, C), generator=g, device=DEV).half()
    go = torch.randint(-1, 2, (5, K), generator=g, device=DEV).half()
    tab = torch.tensor([[3, -1, 0, 4, 2]], dtype=torch.int32, device=DEV)
    dw = conv_backward_weight(x, go, tab, (K, 1, C)).view(K, C)
    o = torch.tensor([0, 2, 3, 4], device=DEV)
    for n0 in range(0, K, 4096):
        ref = go[o, n0:n0 + 4096].float().T.contiguous() @ x[tab[0, o].long()].float()
        assert torch.equal(dw[n0:n0 + 4096], ref.half())
