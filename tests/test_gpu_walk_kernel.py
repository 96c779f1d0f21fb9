"""The fp32 kernel that keeps a block column for several token tiles, against the oracle and, bit for bit, against stream_kernel, which serves calls of a few tokens."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native, workloads
from tests.helpers import assert_close, to64

F32 = torch.float32


def _blocks(out_f, in_f, nnz, zipf, seed):
    grid = out_f // 32, in_f // 32
    if zipf:
        where = workloads.zipf_positions(*grid, nnz, seed=seed)
    else:
        where = np.random.RandomState(seed).permutation(grid[0] * grid[1])[:nnz]
    return [(int(p) // grid[1], int(p) % grid[1]) for p in where]


@pytest.mark.parametrize("n, k, tokens, nnz", [
    (2656, 672, 922, 247), (1856, 768, 2528, 132),   # 0.65 and 0.69 times as fast where columns are uneven: a full one would take most of the launch
    (960, 672, 5473, 137),   # 0.86 (stream_kernel in tiles of 32 tokens)
    (3200, 3488, 5163, 610), (4064, 2240, 2323, 693), (2144, 2880, 10753, 374),   # 0.77 to 0.85: a long one, more than that of its work
])
@pytest.mark.parametrize("transpose", [False, True])
def test_columns_that_may_be_long(n, k, tokens, nnz, transpose):
    """The host does not know how uneven columns are: what loses with uneven ones stays with stream_kernel."""
    assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, F32, False) == "stream_kernel"


@pytest.mark.gpu
@pytest.mark.parametrize("n, k, tokens, nnz, transpose, zipf", [
    (3808, 384, 13134, 72, True, False),        # columns without blocks
    (640, 448, 14976, 129, True, False),
    (1792, 256, 13092 - 13092 % 32, 70, False, False),   # whole tiles only
    (1792, 256, 13092 - 13092 % 32 + 1, 70, True, False),  # one token in the last tile
    (1248, 608, 12843, 75, False, False),
    (1088, 480, 9000, 120, True, True),         # uneven columns
    (1984, 992, 4001, 480, False, False),
    (3072, 1024, 14000, 450, True, False),      # the longest contraction
    (3072, 1024, 14001, 450, False, True),
])
@pytest.mark.parametrize("bias", [False, True])
def test_same_bits_as_stream_kernel(cuda, n, k, tokens, nnz, transpose, zipf, bias):
    assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, F32, False) == "walk_kernel"
    few = 33
    assert native.matmul_kernel_name(few, n, k, nnz, transpose, F32, False) == "stream_kernel"
    torch.manual_seed(nnz)
    shape = (n, k) if transpose else (k, n)
    # (Zipf rows of the matrix are uneven columns of the forward product)
    m = BlockSparseMatrix.zeros(shape, blocks=_blocks(*shape, nnz, zipf, nnz), device="cpu", dtype=F32)
    with torch.no_grad():
        m.data.normal_()
    w = O.to_dense(to64(m.data), m.build_coo_block_index().numpy(), shape)
    w = w.T if transpose else w
    m = m.to(cuda)
    x = torch.randn(tokens, k, device=cuda)
    b = torch.randn(n, device=cuda) if bias else None
    print(n, k, tokens, nnz, transpose, zipf, bias, flush=True)
    ptr, entries = (m.row_start_ends_a, m.cols_a) if transpose else (m.col_start_ends_b, m.rows_b)
    plan = native.blocksparse_matmul_plan(ptr, entries, n, k)
    run = lambda rows: native.blocksparse_matmul(rows, m.data.detach(), plan, n, k, nnz, transpose, bias=b)
    y = run(x)
    assert torch.isfinite(y).all()
    for lo in (0, 31, tokens // 2, tokens - few):
        assert torch.equal(y[lo:lo + few], run(x[lo:lo + few].clone())), lo
    rows = np.r_[0:64, tokens - 64:tokens]
    ref = to64(x[rows]) @ w + (to64(b) if bias else 0.0)
    assert_close(y[rows], ref, F32, "rows at either end")
