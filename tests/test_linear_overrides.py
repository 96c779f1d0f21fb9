"""What a program puts in the place of the layer's parts is called: products of a subclass of the matrix, and `fn`."""
import copy

import numpy as np
import pytest
import torch
import torch.nn.utils.parametrize

from pytorch_block_sparse_amd import BlockSparseLinear, BlockSparseMatrix


class DenseProducts(BlockSparseMatrix):
    """The three products by dense torch operations, the data behind a view."""

    def get_differentiable_data(self):
        return self.data * 1.0

    def reverse_matmul(self, dense_a, transpose, bias=None):
        w = self.to_dense()
        y = dense_a @ (w.t() if transpose else w)
        return y if bias is None else y + bias

    def matmul_with_output_sparse_support(self, dense_a, dense_b, overwrite_data=False):
        w = dense_a.reshape(-1, self.shape[0]).t() @ dense_b.reshape(-1, self.shape[1])
        at = self.build_coo_block_index().long()
        return w.reshape(self.shape[0] // 32, 32, -1, 32).permute(0, 2, 3, 1)[at[0], at[1]].reshape(-1, 32)


def test_products_of_a_subclass():
    np.random.seed(1)
    layer = BlockSparseLinear(96, 64, density=0.5, device="cpu")
    layer.weight = DenseProducts.randn((64, 96), 3, device="cpu")
    x = torch.randn(5, 96, requires_grad=True)
    y = layer(x)
    w = layer.weight.to_dense()
    assert torch.allclose(y, x @ w.t() + layer.bias)
    y.sum().backward()
    assert torch.allclose(x.grad, torch.ones(5, 64) @ w)
    assert layer.weight.data.grad.abs().sum() > 0


def test_replaced_function():
    layer = BlockSparseLinear(96, 64, density=0.5, device="cpu")
    layer.fn = lambda x, data, weight, bias: (x, data, weight, bias)
    x = torch.randn(5, 96)
    got = layer(x)
    assert got[0] is x and got[1] is layer.weight.data and got[2] is layer.weight and got[3] is layer.bias


@pytest.mark.gpu
def test_copies_keep_the_native_path(cuda, monkeypatch):
    layer = copy.deepcopy(BlockSparseLinear(96, 64, density=0.5, device=cuda))
    calls = []
    monkeypatch.setattr(BlockSparseMatrix, "reverse_matmul", lambda *a, **k: calls.append(a))
    assert layer(torch.randn(5, 96, device=cuda)).shape == (5, 64) and not calls


@pytest.mark.gpu
def test_tensors_that_are_not_in_the_dicts(cuda):
    """A parametrized bias, one kept as a plain attribute, and swapped tensors reach the product."""
    np.random.seed(1)
    x = torch.randn(5, 96, device=cuda)

    def plain(layer):
        return x @ layer.weight.to_dense().t()

    layer = BlockSparseLinear(96, 64, density=0.5, device=cuda)
    torch.nn.utils.parametrize.register_parametrization(layer, "bias", type("One", (torch.nn.Module,), {"forward": lambda self, b: b + 1})())
    assert torch.allclose(layer(x), plain(layer) + 1, atol=1e-5)
    layer = BlockSparseLinear(96, 64, density=0.5, device=cuda)
    del layer.bias
    layer.bias = torch.full((64,), 3.0, device=cuda)
    assert torch.allclose(layer(x), plain(layer) + 3, atol=1e-5)
    layer = BlockSparseLinear(96, 64, density=0.5, device=cuda)
    swapped = {"bias": torch.full((64,), 2.0, device=cuda), "weight.data": layer.weight.data.detach() * 2}
    assert torch.allclose(torch.func.functional_call(layer, swapped, (x,)), 2 * plain(layer) + 2, atol=1e-5)
