"""The products of ``native`` on plain tensors and plans, against those of a matrix: the same bits."""
import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native


def test_they_run_on_a_gpu_only():
    t, i = torch.zeros(32, 32), torch.zeros(2, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="run only on a GPU"):
        native.blocksparse_matmul(t, t, i, 32, 32, 1, True)
    with pytest.raises(RuntimeError, match="run only on a GPU"):
        native.blocksparse_matmul_back(t, t, i, i.view(1, 2), t)
    native.check_protocol("nothing to check without PBS_DEBUG")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, tokens, out_f, in_f, blocks", [
    (torch.float32, 33, 256, 96, 20),
    (torch.bfloat16, 4100, 768, 512, 100),
    (torch.bfloat16, 16384, 2048, 2048, 2048),   # with the transposed copy of the blocks; rectangles
])
def test_same_as_the_matrix(cuda, monkeypatch, dtype, tokens, out_f, in_f, blocks):
    monkeypatch.setenv("PBS_DEBUG", "1")
    np.random.seed(blocks)
    torch.manual_seed(blocks)
    m = BlockSparseMatrix.randn((out_f, in_f), blocks, device=cuda, dtype=dtype)
    x, dy, bias = (torch.randn(*s, device=cuda).to(dtype) for s in ((tokens, in_f), (tokens, out_f), (out_f,)))
    data = m.data.detach()
    forward = native.blocksparse_matmul_plan(m.row_start_ends_a, m.cols_a, out_f, in_f)
    y = native.blocksparse_matmul(x, data, forward, out_f, in_f, blocks, True, bias=bias)
    assert torch.equal(y, m.reverse_matmul(x, True, bias=bias))
    back = native.blocksparse_matmul_plan(m.col_start_ends_b, m.rows_b, in_f, out_f)
    out = torch.empty_like(x)
    assert native.blocksparse_matmul(dy, data, back, in_f, out_f, blocks, False, out=out) is out
    assert torch.equal(out, m.reverse_matmul(dy, False))
    dw = native.blocksparse_matmul_back(dy, x, m.row_start_ends_a, m.cols_a, torch.empty_like(data))
    assert torch.equal(dw, m.matmul_with_output_sparse_support(dy, x))
