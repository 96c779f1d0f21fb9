"""The bf16 dense x block-sparse kernels that keep their token tile in LDS, against the CPU oracle, at the sizes where their
tiles of 64 tokens have an edge: whole contractions (rows padded to 128 features, 16 waves' turns through the block columns, two columns'
lists at a time) and contractions in chunks of 512 features (4, 2 or 1 waves per column, lists read 64 entries at a time)."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize(
    "kernel, in_f, out_f, tokens, blocks",
    [
        ("panel_kernel", 768, 3072, 2317, 1152),    # ragged tokens, one column per wave
        ("panel_kernel", 992, 2016, 4097, 900),     # features no multiple of 128 or 64, one token in the last tile
        ("panel_kernel", 1024, 4096, 4096, 1300),   # the longest contraction
        ("panel_kernel", 256, 4096, 16385, 1000),   # several columns per wave
        ("panel_kernel", 256, 4064, 16400, 300),    # columns without blocks, an odd number of columns
        ("panel_kernel", 32, 4096, 40000, 128),     # one k-block, one row piece
        ("panel_kernel", 768, 2048, 8229, 1536),    # every block: full columns
        ("panel_chunk_kernel", 3072, 768, 2317, 1152),     # four waves per column
        ("panel_chunk_kernel", 1056, 544, 4099, 280),      # a last chunk of one k-block, fewer columns than places
        ("panel_chunk_kernel", 4096, 4096, 1024, 4096),    # two waves per column
        ("panel_chunk_kernel", 2048, 2048, 4093, 819),     # one wave per column
        ("panel_chunk_kernel", 4160, 512, 5000, 2080),     # full columns of 130 blocks
    ],
)
def test_edges_against_oracle(cuda, kernel, in_f, out_f, tokens, blocks):
    print(f"{in_f}->{out_f} tokens={tokens} blocks={blocks}", flush=True)
    g = torch.Generator().manual_seed(blocks)
    np.random.seed(blocks)
    x = torch.randn((tokens, in_f), generator=g).to(BF16)
    rows = torch.cat([torch.arange(70), torch.randint(0, tokens, (150,), generator=g), torch.arange(tokens - 70, tokens)])
    for transpose in (True, False):
        shape = (out_f, in_f) if transpose else (in_f, out_f)
        m = BlockSparseMatrix.randn(shape, blocks, device="cpu", dtype=BF16).to(cuda)
        w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), shape)
        assert native.matmul_kernel_name(tokens, out_f, in_f, blocks, transpose, BF16) == kernel
        for bias in (None, torch.randn((out_f + 1,), generator=g).to(BF16)[1:]):   # (a bias that is aligned to two bytes only)
            y = m.reverse_matmul(x.to(cuda), transpose, bias=None if bias is None else bias.to(cuda))
            want = to64(x[rows]) @ (w.T if transpose else w)
            assert_close(y[rows.to(cuda)], want if bias is None else want + to64(bias)[None, :], BF16, f"transpose={transpose} bias={bias is not None}")


def test_chunks_with_empty_columns(cuda):
    """3072 -> 1024, 2317 tokens: the result's first five block columns hold nothing, others 48 blocks."""
    shape = (1024, 3072)
    blocks = [(r, c) for r in range(5, 32) for c in range(96) if (3 * r + c) % 2 == 0]
    m = BlockSparseMatrix.zeros(shape, blocks=blocks, device=cuda, dtype=BF16)
    g = torch.Generator().manual_seed(5)
    with torch.no_grad():
        m.data.copy_(torch.randn(m.data.shape, generator=g))
    x, bias = torch.randn((2317, 3072), generator=g).to(BF16), torch.randn((1024,), generator=g).to(BF16)
    assert native.matmul_kernel_name(2317, 1024, 3072, len(blocks), True, BF16) == "panel_chunk_kernel"
    y = m.reverse_matmul(x.to(cuda), True, bias=bias.to(cuda))
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), shape)
    assert_close(y, to64(x) @ w.T + to64(bias)[None, :], BF16, "empty columns")
