"""The fp32 kernel on the bf16 cores where its groups of eight block columns are far from full: 9, 10 and 17 columns."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu
F32 = torch.float32


@pytest.mark.parametrize("n, k, tokens, nnz, transpose", [
    (288, 1472, 15776, 302, True),
    (320, 2560, 7623, 516, False),
    (544, 1440, 6870, 571, True),
])
def test_groups_with_few_columns(cuda, n, k, tokens, nnz, transpose):
    assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, F32) == "split_kernel"
    np.random.seed(nnz)
    torch.manual_seed(nnz)
    shape = (n, k) if transpose else (k, n)
    m = BlockSparseMatrix.randn(shape, nnz, device="cpu", dtype=F32).to(cuda)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), shape)
    x = torch.randn(tokens, k)
    print(n, k, tokens, nnz, flush=True)
    y = m.reverse_matmul(x.to(cuda), transpose=transpose)
    rows = np.r_[0:300, tokens - 300:tokens]
    ref = to64(x[rows]) @ (w.T if transpose else w)
    assert_close(y[rows], ref, F32, "rows at either end")
    # a block's sum is rounded a few times and joins the total with one rounding, of some 80 blocks at most: sqrt(80) / 2 roundings of 2^-24, halved by their growth with the sum
    assert np.linalg.norm(to64(y[rows].cpu()) - ref) <= 2.5e-7 * np.linalg.norm(ref)
