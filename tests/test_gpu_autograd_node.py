"""The native autograd node of the linear layer under torch's other machinery: forward mode, tracing, hooks on saved tensors
and create_graph."""
import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwad

from pytorch_block_sparse_amd import BlockSparseLinear


def test_forward_mode_is_refused():
    """The layer has no forward-mode derivative: a tangent is refused, not dropped."""
    layer = BlockSparseLinear(64, 64, device="cpu")
    with fwad.dual_level():
        x = fwad.make_dual(torch.randn(4, 64), torch.randn(4, 64))
        with pytest.raises(NotImplementedError, match="forward-mode"):
            layer(x)


def _layer(cuda, n_in=256, n_out=128, dtype=torch.float32):
    np.random.seed(5)
    torch.manual_seed(5)
    layer = BlockSparseLinear(n_in, n_out, density=0.5, device=cuda, dtype=dtype)
    with torch.no_grad():
        layer.bias.normal_()
    return layer


@pytest.mark.gpu
def test_trace_replays_the_layer(cuda):
    layer = _layer(cuda)
    traced = torch.jit.trace(layer, torch.randn(33, 256, device=cuda), check_trace=False)
    x = torch.randn(33, 256, device=cuda)
    assert torch.equal(traced(x), layer(x))


@pytest.mark.gpu
def test_saved_tensor_hooks_and_create_graph(cuda):
    layer = _layer(cuda)
    x = torch.randn(33, 256, device=cuda, requires_grad=True)
    dy = torch.randn(33, 128, device=cuda, requires_grad=True)
    inputs = (x, layer.weight.data, layer.bias)
    plain = torch.autograd.grad(layer(x), inputs, dy.detach())
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.to(cuda)):
        y = layer(x)
    assert sorted(map(tuple, seen)) == sorted([tuple(x.shape), tuple(layer.weight.data.shape)])
    for got, want in zip(torch.autograd.grad(y, inputs, dy.detach()), plain):
        assert torch.equal(got, want)
    # the bias gradient is the sum of dy, whose derivative is one
    db = torch.autograd.grad(layer(x), layer.bias, dy, create_graph=True)[0]
    assert torch.equal(torch.autograd.grad(db.sum(), dy)[0], torch.ones_like(dy))
