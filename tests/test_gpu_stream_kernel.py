"""The dense x block-sparse kernel with one block column per workgroup, against the CPU oracle, at the sizes where its
token tiles (16 to 128 tokens), its waves' turns through a column's blocks (2 to 8 waves, lists of more than 64 blocks per
wave) and its split over the XCDs have an edge."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(
    "in_f, out_f, tokens, blocks",
    [
        (32, 32, 1, 1),            # one block, one token
        (96, 64, 17, 3),           # contraction no multiple of 64, one token into the second tile
        (2560, 256, 15, 400),      # long columns over few tokens
        (320, 1312, 129, 90),      # short columns (some empty), 128 tokens and one
        (256, 288, 4099, 36),      # many token tiles, fewer columns than XCDs x 2
        (8736, 32, 70, 273),       # one full column of 273 blocks: over 64 per wave
        (640, 96, 1023, 41),
    ],
)
def test_edges_against_oracle(cuda, dtype, in_f, out_f, tokens, blocks):
    print(f"{in_f}->{out_f} tokens={tokens} blocks={blocks} {dtype}", flush=True)
    np.random.seed(blocks)
    torch.manual_seed(blocks)
    m = BlockSparseMatrix.randn((out_f, in_f), blocks, device="cpu", dtype=dtype).to(cuda)
    x, dy, bias = (torch.randn(*s).to(dtype) for s in ((tokens, in_f), (tokens, out_f), (out_f,)))
    w = O.to_dense(to64(m.data), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    for n, k, transpose in ((out_f, in_f, True), (in_f, out_f, False)):
        assert native.matmul_kernel_name(tokens, n, k, blocks, transpose, dtype) == "stream_kernel"
    y = m.reverse_matmul(x.to(cuda), True, bias=bias.to(cuda))
    assert_close(y, to64(x) @ w.T + to64(bias)[None, :], dtype, "forward")
    assert_close(m.reverse_matmul(dy.to(cuda), False), to64(dy) @ w, dtype, "input gradient")


def test_result_of_a_token_does_not_depend_on_the_others(cuda):
    """fp32: one order of summation per pattern, whatever tile the token count leads to."""
    torch.manual_seed(3)
    np.random.seed(3)
    for in_f, out_f, blocks in ((768, 512, 200), (768, 512, 60)):
        m = BlockSparseMatrix.randn((out_f, in_f), blocks, device=cuda)
        x = torch.randn(5000, in_f, device=cuda)
        y = m.reverse_matmul(x, True)
        for lo, hi in ((0, 1), (77, 300), (4000, 5000)):
            assert torch.equal(m.reverse_matmul(x[lo:hi], True), y[lo:hi])
