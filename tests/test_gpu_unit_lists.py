"""The lists of units of the row weight gradient: at most one to six blocks of a block row per workgroup.  Each list holds every block once, and the
kernels are right with each, in one slice of the tokens and in several, with a table from the caller and with one made in the workspace."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16


def _p(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None and t.numel() else 0)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _matrix(cuda, out_f, in_f, nnz, dtype=F32):
    np.random.seed(nnz)
    return BlockSparseMatrix.randn((out_f, in_f), nnz, device=cuda, dtype=dtype)


@pytest.mark.parametrize("out_f, in_f, nnz", [(96, 416, 17), (3072, 768, 1050), (416, 160, 1), (32 * 1024, 64, 300), (64, 64, 0)])
def test_every_list_holds_every_block_once(cuda, out_f, in_f, nnz):
    m = _matrix(cuda, out_f, in_f, nnz)
    lib, rows = native.load(), out_f // 32
    size = lib.pbs_blocksparse_matmul_back_units_bytes(64, out_f, in_f, nnz, 0)
    table = torch.full((size // 4,), -7, dtype=torch.int32, device=cuda)
    assert lib.pbs_blocksparse_matmul_back_units(_p(m.row_start_ends_a), _p(m.cols_a), out_f, in_f, nnz, _p(table), size, _stream()) == 0
    table = table.cpu().numpy()
    coo = m.build_coo_block_index().cpu().numpy() if nnz else np.zeros((2, 0), int)
    want = sorted((int(r), int(c), b) for b, (r, c) in enumerate(coo.T))
    counts, at = np.bincount(coo[0], minlength=rows), 16
    for per_unit in range(1, 7):
        units = table[at:at + 16 * table[per_unit - 1]].reshape(-1, 16)
        assert len(units) == sum(max(1, -(-n // per_unit)) for n in counts)
        got = [(u[0], u[4 + i], u[10 + i]) for u in units for i in range(u[1])]
        assert sorted(got) == want and (len(units) == 0 or units[:, 1].max() <= per_unit)
        first = [u[0] for u in units if u[2] == 0]   # the unit of a row that sums its bias gradient
        assert sorted(first) == list(range(rows))
        at += 16 * (nnz // per_unit + rows)
    assert at == len(table)


@pytest.mark.parametrize("dtype, per_unit, slices, tokens, out_f, in_f, nnz", [
    (F32, 1, 1, 33, 416, 160, 3), (F32, 2, 1, 33, 3072, 768, 239), (F32, 3, 1, 33, 3072, 416, 449), (F32, 4, 1, 33, 3072, 416, 643),
    (F32, 5, 1, 33, 3072, 416, 842), (F32, 6, 1, 33, 3072, 768, 1050),
    (F32, 1, 2, 1500, 416, 160, 3), (F32, 2, 2, 2317, 3072, 160, 25), (F32, 3, 2, 3000, 416, 768, 76), (F32, 4, 2, 2317, 416, 416, 62),
    (F32, 5, 2, 3000, 2048, 416, 113), (F32, 6, 2, 2317, 416, 992, 256),
    # sdd_split_kernel: 2^20 tokens x blocks and more
    (F32, 2, 1, 1500, 2912, 320, 906), (F32, 2, 2, 4097, 3072, 128, 262), (F32, 3, 1, 1500, 800, 928, 707), (F32, 3, 2, 3000, 160, 2496, 353),
    (F32, 4, 1, 700, 1248, 1248, 1503), (F32, 4, 2, 1500, 2112, 352, 723),
    (BF16, 1, 1, 33, 416, 160, 3), (BF16, 2, 1, 33, 3072, 160, 197), (BF16, 3, 1, 33, 3072, 768, 464), (BF16, 4, 1, 33, 3072, 416, 673),
    (BF16, 5, 1, 33, 3072, 768, 881), (BF16, 6, 1, 33, 3072, 416, 1092),
    (BF16, 1, 2, 2317, 416, 160, 3), (BF16, 2, 2, 2317, 416, 160, 21), (BF16, 3, 2, 3000, 2048, 160, 17), (BF16, 4, 2, 3000, 1024, 160, 60),
    (BF16, 5, 2, 3000, 1024, 160, 120), (BF16, 6, 2, 3000, 1504, 160, 92),
])
def test_kernels_with_every_list(cuda, dtype, per_unit, slices, tokens, out_f, in_f, nnz):
    """`slices` 2: several."""
    lib, code = native.load(), native.DTYPE_CODES[dtype]
    kernel = "sdd_split_kernel" if dtype == F32 and tokens * nnz >= 1 << 20 else "sdd_row_kernel"
    assert native.matmul_back_kernel_name(tokens, out_f, in_f, nnz, dtype) == (kernel if slices == 1 else kernel + " + sdd_reduce_kernel")
    size = lib.pbs_blocksparse_matmul_back_workspace_bytes(tokens, out_f, in_f, nnz, code)
    partial = size - 64 - (nnz // per_unit + out_f // 32) * 64   # what the list of these units leaves
    assert partial % (nnz * 4096) == 0 and (partial > 0) == (slices > 1)
    m = _matrix(cuda, out_f, in_f, nnz, dtype)
    torch.manual_seed(tokens)
    x, dy = torch.randn(tokens, in_f, device=cuda).to(dtype), torch.randn(tokens, out_f, device=cuda).to(dtype)
    at = m.build_coo_block_index().long()
    dense = dy.double().t().contiguous() @ x.double()
    want = dense.reshape(out_f // 32, 32, in_f // 32, 32).permute(0, 2, 3, 1)[at[0], at[1]].reshape(-1, 32)
    print(dtype, per_unit, slices, tokens, out_f, in_f, nnz, flush=True)
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(x, data, bias, m._buffers, m.schedule()).backward(dy)
    plain = torch.full_like(data.grad, float("nan"))
    ws = torch.full((size,), 0x7f, dtype=torch.uint8, device=cuda)
    assert lib.pbs_blocksparse_matmul_back(_p(dy), _p(x), _p(m.row_start_ends_a), _p(m.cols_a), _p(plain), tokens, out_f, in_f, nnz, code, _p(ws), size, _stream()) == 0
    assert torch.equal(plain, data.grad)
    # fp32: a chunk's chain of 32 terms, at most 12 chunks or groups of 8 of them one behind the other, four waves and the slices: fewer than 64 roundings of
    # 2^-25 on average, in a random walk over half of them; bf16: one rounding of the result, 2^-9 at most
    limit = 64 ** 0.5 * 2.0 ** -25 if dtype == F32 else 2.0 ** -9
    assert (data.grad.double() - want).norm() <= limit * want.norm()
    assert (bias.grad.double() - dy.double().sum(0)).norm() <= limit * dy.double().sum(0).norm()
