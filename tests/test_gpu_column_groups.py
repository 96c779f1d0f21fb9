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
    ("wide", 1536, 128, 128 * 86 + 5),
    ("wide", 3584, 64, 128 * 37),
])
def test_every_tile_of_every_group(cuda, monkeypatch, kernel, out_f, in_f, tokens):
    monkeypatch.setenv("PBS_COLUMN_KERNEL", "1" if kernel == "column" else "0")
    nnz = out_f // 32
    assert native.matmul_kernel_name(tokens, out_f, in_f, nnz, True, BF16, kernel == "column") == ("ddsc_kernel" if kernel == "column" else "dds16_kernel")
    np.random.seed(out_f)
    torch.manual_seed(out_f)
    m = BlockSparseMatrix.randn((out_f, in_f), nnz, device="cpu", dtype=BF16).to(cuda)
    x = torch.randn(tokens, in_f).to(BF16)
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    print(kernel, out_f, in_f, tokens, flush=True)
    assert_close(m.reverse_matmul(x.to(cuda), transpose=True), to64(x) @ w.T, BF16, "forward")
