"""The lists of both directions and the units of the weight gradient, derived in one launch, against the calls that make them one
by one: the same bytes."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_f, in_f, blocks", [
    (32, 32, 1),
    (3072, 768, 1152),
    (96, 4096, 50),            # rows without blocks in one direction, columns without in the other
    (4096, 4096, 5000),
    (32 * 1500, 64, 700),      # more rows than the units' prefix sum holds in LDS
    (64, 32 * 9000, 300),      # more columns than are ranked
    (128, 128, 0),
])
@pytest.mark.parametrize("with_units", [True, False])
def test_same_bytes_as_one_by_one(cuda, out_f, in_f, blocks, with_units):
    np.random.seed(blocks)
    m = BlockSparseMatrix.randn((out_f, in_f), blocks, device=cuda)
    lib = native.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None and t.numel() else 0)
    sizes = (lib.pbs_blocksparse_matmul_plan_bytes(out_f, in_f), lib.pbs_blocksparse_matmul_plan_bytes(in_f, out_f),
             lib.pbs_blocksparse_matmul_back_units_bytes(64, out_f, in_f, blocks, 0))
    one, all_ = ([torch.zeros(n, dtype=torch.uint8, device=cuda) for n in sizes] for _ in range(2))
    part = lib.pbs_blocksparse_matmul_plan_part
    assert part(p(m.row_start_ends_a), p(m.cols_a), out_f, in_f, blocks, 1, p(one[0]), sizes[0], stream) == 0
    assert part(p(m.col_start_ends_b), p(m.rows_b), in_f, out_f, blocks, 1, p(one[1]), sizes[1], stream) == 0
    if with_units:
        assert lib.pbs_blocksparse_matmul_back_units(p(m.row_start_ends_a), p(m.cols_a), out_f, in_f, blocks, p(one[2]), sizes[2], stream) == 0
    assert lib.pbs_blocksparse_derive(p(m.row_start_ends_a), p(m.cols_a), p(m.col_start_ends_b), p(m.rows_b), out_f, in_f, blocks,
                                      p(all_[0]), sizes[0], p(all_[1]), sizes[1], p(all_[2]) if with_units else None, sizes[2], stream) == 0
    torch.cuda.synchronize()
    for a, b in zip(one, all_):
        assert torch.equal(a, b)
