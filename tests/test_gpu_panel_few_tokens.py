"""bf16 products of 768 to 1023 tokens in chunks of a shared token tile (panel_chunk_kernel), and their neighbours that stay in the stream kernel."""
import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transpose", [True, False])
@pytest.mark.parametrize("tokens, k, n, nnz, chunks", [
    (1015, 2720, 4064, 5408, True), (769, 4064, 2720, 5408, True), (1023, 2048, 3072, 4000, True), (896, 4096, 1536, 3000, True),
    (767, 2720, 4064, 5408, False), (1015, 2016, 4064, 4000, False), (1015, 4096, 1504, 3000, False), (1015, 4064, 4096, 16 * 128 - 1, False),
])
def test_few_tokens(cuda, tokens, k, n, nnz, chunks, transpose):
    kernel = native.load().pbs_blocksparse_matmul_kernel_name(tokens, n, k, nnz, int(transpose), 1, 1).decode()
    assert (kernel == "panel_chunk_kernel") == chunks, kernel
    np.random.seed(tokens)
    m = BlockSparseMatrix.randn((n, k) if transpose else (k, n), nnz, device=cuda, dtype=torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    a = torch.randn((tokens, k), generator=g, device=cuda).bfloat16()
    got, dense = m.reverse_matmul(a, transpose=transpose), m.to_dense().double()
    dense = (dense.t() if transpose else dense).contiguous()
    want, most = a.double() @ dense, a.double().abs() @ dense.abs()
    # one rounding of the result to bf16, and sums of at most k products in fp32
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + k * 2.0 ** -24 * most).all())
