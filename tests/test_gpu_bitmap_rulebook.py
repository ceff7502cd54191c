"""Rulebooks of strided and transposed convolutions from the occupancy bitmap, at
the sizes where its scan and its window instances can go wrong: one word, a
chunk's last word, more chunks than the scan looks back over at once, windows of
3 and more offsets, missing leading dimensions, dilation, and a bound that cuts
the outputs."""

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# shape, kernel, stride, padding, dilation, transpose, rows
CASES = [
    ([5], [3], [1], [1], [1], False, 4),  # a single word
    ([262144], [3], [1], [1], [1], False, 900),  # one whole chunk of the scan
    ([262145], [2], [1], [0], [1], False, 900),
    ([700, 900], [3, 2], [2, 1], [1, 0], [1, 2], False, 2000),  # two dimensions
    ([64, 512, 640], [3, 3, 3], [1, 1, 1], [1, 1, 1], [1, 1, 1], False, 6000),  # 80 chunks
    ([64, 256, 320], [3, 1, 2], [2, 1, 2], [1, 0, 0], [1, 1, 1], True, 6000),
    ([24, 40, 40], [3, 3, 3], [2, 2, 2], [1, 1, 1], [2, 1, 17], False, 3000),  # words far apart
    ([24, 40, 40], [5, 3, 3], [2, 2, 2], [2, 1, 1], [1, 1, 1], False, 3000),  # general windows
    ([6, 10, 12, 12], [3, 3, 3, 3], [2, 2, 2, 2], [1, 1, 1, 1], [1, 1, 1, 1], False, 2000),
]


@pytest.mark.parametrize("ci", range(len(CASES)))
def test_bitmap_rulebook_matches_oracle(ci):
    from spconv_triton.core import ConvAlgo
    from spconv_triton.pytorch import ops

    shape, ks, st, pad, dil, tr, n = CASES[ci]
    nd = len(shape)
    rng = np.random.default_rng(7000 + ci)
    lin = rng.choice(2 * int(np.prod(shape)), size=n, replace=False)
    idx = np.stack(np.unravel_index(lin, [2] + shape), 1).astype(np.int32)
    it = torch.from_numpy(idx).to(DEV)
    exp = orc.igemm_pairs(idx, 2, shape, ks, st, pad, dil, [0] * nd, False, tr, True)
    for bound in (-1, max(1, exp[0].shape[0] // 3)):
        res = ops.get_indice_pairs_implicit_gemm(
            it, 2, shape, ConvAlgo.MaskImplicitGemm, ks, st, pad, dil, [0] * nd, False, tr,
            is_train=True, num_out_act_bound=bound)
        m = exp[0].shape[0] if bound < 0 else bound
        np.testing.assert_array_equal(res[0].cpu().numpy(), exp[0][:m])
        np.testing.assert_array_equal(res[2].cpu().numpy(), exp[2][:, :m])
        bwd = np.where(exp[3] < m, exp[3], -1)
        np.testing.assert_array_equal(res[3].cpu().numpy(), bwd)
        assert int((res[2] >= 0).sum()) == int((bwd >= 0).sum())


def test_rulebooks_of_many_threads_at_once():
    """Each call in flight has its own counts, whatever the thread, stream or size."""
    import threading

    from spconv_triton.core import ConvAlgo
    from spconv_triton.pytorch import ops

    rng = np.random.default_rng(11)
    shape = [16, 40, 48]

    def build(it):
        return ops.get_indice_pairs_implicit_gemm(
            it, 1, shape, ConvAlgo.MaskImplicitGemm, [3] * 3, [2] * 3, [1] * 3, [1] * 3, [0] * 3,
            False, False, is_train=True)

    inputs, want = [], []
    for n in (5, 90, 400, 1500, 3000, 4000, 6000, 9000):
        lin = np.sort(rng.choice(int(np.prod(shape)), size=n, replace=False))
        idx = np.concatenate([np.zeros((n, 1)), np.stack(np.unravel_index(lin, shape), 1)], 1)
        inputs.append(torch.from_numpy(idx.astype(np.int32)).to(DEV))
        res = build(inputs[-1])
        want.append([res[0].cpu(), res[2].cpu(), res[3].cpu()])
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    res = build(inputs[i])
                    got = [res[0].cpu(), res[2].cpu(), res[3].cpu()]
                    assert all(torch.equal(a, b) for a, b in zip(got, want[i]))
        except BaseException as e:  # (an assertion in a thread would be lost)
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
