"""fp32 results of 9, 10, 11 and 17 block columns: the kernel on the bf16 cores wants three quarters of the places of its groups filled, so they are the fp32 matrix
instructions', in any number of tokens: what is one product is that product, rounded once, and a token's result has the same bits in any batch."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

F32 = torch.float32


@pytest.mark.parametrize("cols", range(1, 41))
@pytest.mark.parametrize("transpose", [True, False])
def test_filled_groups_only(cols, transpose):
    names = {native.matmul_kernel_name(tokens, 32 * cols, 1472, nnz, transpose, F32)
             for tokens in (700, 4096, 15776) for nnz in range(cols * 46 // 4, cols * 46, cols * 8)}
    groups = -(-cols // 8)
    if 4 * cols < 3 * 8 * groups:
        assert "split_kernel" not in names, names
    elif cols >= 18:
        assert "split_kernel" in names, names


@pytest.mark.gpu
@pytest.mark.parametrize("n, k, tokens, nnz, transpose", [
    (288, 1472, 15776, 302, True),
    (320, 2560, 7623, 516, False),
    (352, 1600, 9001, 400, True),
    (544, 1440, 6870, 571, True),
])
def test_groups_with_few_columns(cuda, n, k, tokens, nnz, transpose):
    np.random.seed(nnz)
    torch.manual_seed(nnz)
    shape = (n, k) if transpose else (k, n)
    m = BlockSparseMatrix.randn(shape, nnz, device="cpu", dtype=F32).to(cuda)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), shape)
    w = w.T if transpose else w
    x = torch.randn(tokens, k)
    one = torch.zeros(tokens, k).scatter_(1, torch.randint(k, (tokens, 1)), torch.randn(tokens, 1))
    print(n, k, tokens, nnz, native.matmul_kernel_name(tokens, n, k, nnz, transpose, F32), flush=True)
    y = m.reverse_matmul(x.to(cuda), transpose=transpose)
    rows = np.r_[0:300, tokens - 300:tokens]
    assert_close(y[rows], to64(x[rows]) @ w, F32, "rows at either end")
    assert torch.equal(y[:33], m.reverse_matmul(x[:33].to(cuda), transpose=transpose))
    # one value to a token: every result is one product, rounded to 24 bits, and zeros
    got, ref = to64(m.reverse_matmul(one.to(cuda), transpose=transpose)[rows]), to64(one[rows]) @ w
    assert (np.abs(got - ref) <= 2.0 ** -24 * np.abs(ref) + 2.0 ** -149).all(), np.abs(got - ref).max() / np.abs(ref).max()
