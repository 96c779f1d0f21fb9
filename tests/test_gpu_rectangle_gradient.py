"""The bf16 weight gradient of larger layers, in rectangles of 16 x 16 or 8 x 16 block positions, against float64: bands and column pairs that
are cut off, one to four passes over the accumulators, rows dealt by their counts, slices that end inside a chunk of 32 tokens."""
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import native
from tests.helpers import assert_close, to64
from tests.test_gpu_row_gradient import _layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,out_f,in_f,counts", [
    (13001, 1056, 1056, [4]),              # sixteen rows; a band of one row, a rectangle of one column
    (13001, 1056, 1056, [12]),             # eight rows, one pass
    (13007, 1056, 1056, [33]),             # dense: two passes
    (13007, 1056, 1056, [30, 2, 2, 2]),    # uneven rows are dealt to the bands
    (2600, 64, 10240, [90]),               # more rectangles than rows, 20 columns each
    (16391, 1600, 512, [7, 0, 3, 16]),
    (800, 512, 33056, [1033, 1020, 1031]),  # eight rows, more entries in a band than its list in LDS holds
    (26001, 544, 544, [17, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0]),   # one row of a band has all the blocks, rectangles without blocks
])
def test_rectangles(cuda, tokens, out_f, in_f, counts):
    dtype = torch.bfloat16
    m = _layer(out_f, in_f, counts, dtype, cuda, 5)
    name = native.matmul_back_kernel_name(tokens, out_f, in_f, m.cols_a.shape[0], dtype)
    print(name, tokens, out_f, in_f, flush=True)
    assert name.startswith("sdd_bf16_kernel")
    g = torch.Generator().manual_seed(tokens)
    x, dy = (torch.randn((tokens, f), generator=g).to(dtype) for f in (in_f, out_f))
    ref = O.matmul_with_output_sparse_support(to64(dy), to64(x), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    xd, dyd = x.to(cuda), dy.to(cuda)
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(xd, data, bias, m._buffers, m.schedule()).backward(dyd)
    assert_close(data.grad, ref, dtype, "weight gradient")
    assert_close(bias.grad, to64(dy).sum(0), dtype, "bias gradient")
    assert torch.equal(m.matmul_with_output_sparse_support(dyd, xd), data.grad)   # without the bias gradient
