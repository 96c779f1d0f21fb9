"""The persistent bf16 kernels over numbers of column groups and token tiles that do not divide the chip: every result element is written, by the workgroup
that has its (token tile, group), whatever share of the groups and of the token streams an XCD is dealt."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


# groups of 16 block columns -> token streams: 1 -> 256, 3 -> 85, 4 -> 64, 5 -> 51, 6 -> 42, 7 -> 36, 8 -> 32, 9 -> 28
@pytest.mark.parametrize("kernel, out_f, in_f, tokens", [
    ("column", 512, 128, 128 * 257 + 1),       # a stream with a tile more than the others, on one XCD
    ("column", 1536, 64, 128 * 86 + 5),
    ("column", 1984, 128, 128 * 63 + 127),     # places without a column, fewer tiles than streams
    ("column", 2560, 128, 128 * 51),           # one tile for each stream
    ("column", 3072, 128, 128 * 50 + 1),
    ("column", 3584, 192, 128 * 37),
    ("column", 3584, 64, 1),                   # one tile: one stream
    ("column", 4096, 128, 128 * 33),
    ("column", 4608, 64, 128 * 30),
    ("column", 2048, 4096, 12300),             # an operand of 100 MB: lines asked for ahead
    ("wide", 1536, 128, 128 * 86 + 5),
    ("wide", 3584, 64, 128 * 37),
])
def test_every_tile_of_every_group(cuda, monkeypatch, kernel, out_f, in_f, tokens):
    monkeypatch.setenv("PBS_COLUMN_KERNEL", "1" if kernel == "column" else "0")
    nnz = out_f // 32 * (8 if in_f == 4096 else 1)
    assert native.matmul_kernel_name(tokens, out_f, in_f, nnz, True, BF16, kernel == "column") == ("ddsc_kernel" if kernel == "column" else "dds16_kernel")
    if in_f == 4096:
        assert native.matmul_kernel_form(tokens, out_f, in_f, nnz, True, BF16).endswith(", lines ahead")
    np.random.seed(out_f)
    torch.manual_seed(out_f)
    # (a group whose columns are uneven does not ask ahead)
    blocks = [(r, (16 * j + r) % 128) for r in range(out_f // 32) for j in range(8)] if in_f == 4096 else None
    m = BlockSparseMatrix.randn((out_f, in_f), None if blocks else nnz, blocks=blocks, device="cpu", dtype=BF16).to(cuda)
    x = torch.randn(tokens, in_f).to(BF16)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    print(kernel, out_f, in_f, tokens, flush=True)
    assert_close(m.reverse_matmul(x.to(cuda), transpose=True), to64(x) @ w.T, BF16, "forward")


@pytest.mark.parametrize("out_f, in_f, tokens, nnz", [
    (1056, 1120, 1, 400),
    (1056, 1120, 300, 35 * 33),      # every block
    (1120, 1056, 128 * 129 + 77, 60),
    (2080, 4000, 128 * 70, 2500),    # lists of more than 64 items
    (1056, 4064, 128 * 70 + 1, 127 * 33),   # every block, in the longest lists: 2032 items of a group in the room for 2048
    (4064, 2080, 300, 2500),
])
def test_odd_numbers_of_k_blocks(cuda, monkeypatch, out_f, in_f, tokens, nnz):
    """The last pair of k-blocks is one k-block: its second half is never multiplied, whatever lies behind the row (here NaN: the next row's start)."""
    monkeypatch.setenv("PBS_COLUMN_KERNEL", "1")
    np.random.seed(nnz)
    torch.manual_seed(nnz)
    m = BlockSparseMatrix.randn((out_f, in_f), nnz, device="cpu", dtype=BF16).to(cuda)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    for transpose, n, k, wt in ((True, out_f, in_f, w.T), (False, in_f, out_f, w)):
        assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, BF16, True) == "ddsc_kernel"
        a = torch.randn(tokens, k).to(BF16)
        a[1::2] = float("nan")
        print(n, k, tokens, nnz, transpose, flush=True)
        got = m.reverse_matmul(a.to(cuda), transpose=transpose)
        assert_close(got[0::2], to64(a[0::2]) @ wt, BF16, "transpose %d" % transpose)


@pytest.mark.parametrize("out_f, in_f, tokens, nnz, transpose", [
    (3744, 3360, 7261, 1230, True),
    (2016, 3936, 15003, 706, True),     # an odd number of k-blocks, 118 MB: lines asked for ahead
    (3072, 1952, 13826, 677, False),
])
def test_operands_that_the_stream_kernel_reads_again(cuda, out_f, in_f, tokens, nnz, transpose):
    """Large dense operands with few blocks to a column go to the column kernel by its estimate; a forward product without a workspace does not."""
    n, k = (out_f, in_f) if transpose else (in_f, out_f)
    assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, BF16, True) == "ddsc_kernel"
    assert native.matmul_kernel_form(tokens, n, k, nnz, transpose, BF16).endswith(", lines ahead") == (out_f == 2016)
    if transpose:
        assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, BF16, False) != "ddsc_kernel"
    np.random.seed(nnz)
    torch.manual_seed(nnz)
    m = BlockSparseMatrix.randn((out_f, in_f), nnz, device="cpu", dtype=BF16).to(cuda)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    a = torch.randn(tokens, k).to(BF16)
    print(n, k, tokens, nnz, transpose, flush=True)
    got = m.reverse_matmul(a.to(cuda), transpose=transpose)
    rows = np.r_[0:260, tokens - 260:tokens]
    assert_close(got[rows], to64(a[rows]) @ (w.T if transpose else w), BF16, "rows at either end")
