"""A plan that is made in parts takes the memory that the products read, and no more."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native


@pytest.mark.parametrize("n, k", [(32, 32), (64, 96), (4096, 4096), (3072, 768), (512, 8192), (1504, 992), (992, 1024),
                                  (1504, 1056), (2080, 4000), (512, 4064), (512, 4128)])
def test_size_of_the_parts(n, k):
    lib = native.load()
    cols, kb = n // 32, k // 32
    lists = (cols + 7) // 8 * (8 * 16 + kb * 8 * 8)
    wide = 0 if kb % 2 else (cols + 15) // 16 * (kb // 2 + 2) * 256 + 1024
    # (an odd number of k-blocks from 1056 features on; the lists of 16 columns of up to 128 blocks)
    column = 0 if kb > 128 or (kb % 2 and k <= 1024) else (cols + 15) // 16 * (64 + (64 + (kb + 1) // 2 + 32 * kb) * 4) + 16384 * 4
    assert lib.pbs_blocksparse_matmul_plan_part_bytes(n, k) == lists + wide + column <= lib.pbs_blocksparse_matmul_plan_bytes(n, k)
    assert lib.pbs_blocksparse_matmul_plan_part_bytes(n, k + 1) == 0
    p = ctypes.c_void_p(0x1000)
    part = lib.pbs_blocksparse_matmul_plan_part
    assert part(p, p, n, k, 1, 1, p, lists + wide + column - 1, None) == -5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, n, k, tokens, blocks", [
    (torch.float32, 256, 96, 33, 20), (torch.bfloat16, 1024, 4096, 16384, 512), (torch.bfloat16, 2048, 2048, 16384, 2048),
])
def test_parts_in_exactly_that_much_memory(cuda, dtype, n, k, tokens, blocks):
    """The parts fill their buffer to the end and nothing behind it; a product with them is that of the whole plan."""
    lib = native.load()
    np.random.seed(blocks)
    torch.manual_seed(blocks)
    m = BlockSparseMatrix.randn((n, k), blocks, device=cuda, dtype=dtype)
    size = lib.pbs_blocksparse_matmul_plan_part_bytes(n, k)
    buffer = torch.full((size + 4096,), 77, dtype=torch.uint8, device=cuda)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.pbs_blocksparse_matmul_plan_part(p(m.row_start_ends_a), p(m.cols_a), n, k, blocks, 7, p(buffer), size, stream) == 0
    assert (buffer[size:] == 77).all()
    whole = native.blocksparse_matmul_plan(m.row_start_ends_a, m.cols_a, n, k)
    x = torch.randn(tokens, k, device=cuda).to(dtype)
    print(native.matmul_kernel_name(tokens, n, k, blocks, True, dtype), flush=True)
    assert torch.equal(native.blocksparse_matmul(x, m.data.detach(), buffer, n, k, blocks, True),
                       native.blocksparse_matmul(x, m.data.detach(), whole, n, k, blocks, True))
