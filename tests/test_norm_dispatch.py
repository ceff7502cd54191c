"""Which BatchNorm1d and ReLU modules SparseSequential may run as one launch: the parts of the
choice that need no GPU."""

import pytest
import torch
from torch import nn


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
