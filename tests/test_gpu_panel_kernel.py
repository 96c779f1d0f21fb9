"""The bf16 dense x block-sparse kernel that keeps its token tile in LDS, against the CPU oracle, at the sizes where its
tiles of 64 tokens, its rows in LDS (padded to 128 features), its waves' turns through the block columns (16 waves, two columns'
lists at a time) and its workgroups per tile have an edge."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize(
    "in_f, out_f, tokens, blocks",
    [
        (768, 3072, 2317, 1152),    # ragged tokens, one column per wave
        (992, 2016, 4097, 900),     # features no multiple of 128 or 64, one token in the last tile
        (1024, 4096, 4096, 1300),   # the longest contraction
        (256, 4096, 16385, 1000),   # several columns per wave
        (256, 4064, 16400, 300),    # columns without blocks, an odd number of columns
        (32, 4096, 40000, 128),     # one k-block, one row piece
        (768, 2048, 8229, 1536),    # every block: full columns
    ],
)
def test_edges_against_oracle(cuda, in_f, out_f, tokens, blocks):
    print(f"{in_f}->{out_f} tokens={tokens} blocks={blocks}", flush=True)
    g = torch.Generator().manual_seed(blocks)
    np.random.seed(blocks)
    x = torch.randn((tokens, in_f), generator=g).to(BF16)
    rows = torch.cat([torch.arange(70), torch.randint(0, tokens, (150,), generator=g), torch.arange(tokens - 70, tokens)])
    for transpose in (True, False):
        shape = (out_f, in_f) if transpose else (in_f, out_f)
        m = BlockSparseMatrix.randn(shape, blocks, device="cpu", dtype=BF16).to(cuda)
        w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), shape)
        assert native.matmul_kernel_name(tokens, out_f, in_f, blocks, transpose, BF16) == "panel_kernel"
        for bias in (None, torch.randn((out_f + 1,), generator=g).to(BF16)[1:]):   # (a bias that is aligned to two bytes only)
            y = m.reverse_matmul(x.to(cuda), transpose, bias=None if bias is None else bias.to(cuda))
            want = to64(x[rows]) @ (w.T if transpose else w)
            assert_close(y[rows.to(cuda)], want if bias is None else want + to64(bias)[None, :], BF16, f"transpose={transpose} bias={bias is not None}")
