"""The layer's native autograd node under compiled autograd, against its ordinary backward pass: bit for bit."""
import numpy as np
import pytest
import torch
from torch._dynamo import compiled_autograd

from pytorch_block_sparse_amd import BlockSparseLinear

pytestmark = pytest.mark.gpu


def _layer(cuda, seed, bias=True):
    np.random.seed(seed)
    torch.manual_seed(seed)
    return BlockSparseLinear(256, 128, bias=bias, density=0.5, device=cuda)


def _gradients(layer, x, dy, compiler=None):
    leaves = [t for t in (x, *layer.parameters()) if t.requires_grad]
    for t in leaves:
        t.grad = None
    y = layer(x)
    if compiler is None:
        y.backward(dy)
    else:
        with compiled_autograd._enable(compiler):
            y.backward(dy)
    return [t.grad.clone() for t in leaves]


@pytest.mark.parametrize("compiler", [lambda graph: graph, torch.compile(backend="eager", dynamic=True)], ids=["graph", "dynamo"])
def test_same_gradients(cuda, compiler):
    """Two patterns of one size, with and without bias, input and weight gradient, several token counts: a graph made for one of
    them must not serve another."""
    layers = [_layer(cuda, 1), _layer(cuda, 2), _layer(cuda, 3, bias=False)]
    frozen = _layer(cuda, 4)
    frozen.weight.requires_grad_(False)
    layers.append(frozen)
    for tokens in (33, 33, 64, 5):
        for i, layer in enumerate(layers):
            for wants_x in (True, False):
                if not wants_x and layer is frozen:
                    continue
                print(tokens, i, wants_x, flush=True)
                x = torch.randn(3, tokens, 256, device=cuda, requires_grad=wants_x)
                dy = torch.randn(3, tokens, 128, device=cuda)
                want = _gradients(layer, x, dy)
                got = _gradients(layer, x, dy, compiler)
                assert len(got) == len(want) and all(map(torch.equal, got, want))


def test_new_pattern_between_steps(cuda):
    layer = _layer(cuda, 5)
    x, dy = torch.randn(33, 256, device=cuda, requires_grad=True), torch.randn(33, 128, device=cuda)
    free = (~layer.weight.block_mask_build(None)).nonzero()
    for step in range(3):
        want = _gradients(layer, x, dy)
        got = _gradients(layer, x, dy, lambda graph: graph)
        assert all(map(torch.equal, got, want)), step
        layer.weight.block_replace(torch.cat([free[step:step + 1], torch.tensor([[step]], device=cuda)], 1))
