"""The bf16 weight gradient in more rectangles than there have to be: bands of equal numbers of rows, in pairs, and columns dealt to more rectangles, against float64."""
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import native
from tests.helpers import assert_close, to64
from tests.test_gpu_row_gradient import _layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,out_f,in_f,counts,partition", [
    (13007, 992, 1056, [24], "4 even bands of 8 rows x 4 rectangles"),            # a rectangle more in each band; odd numbers of rows and of columns
    (13007, 992, 1504, [47], "8 even bands of 8 rows x 3 rectangles"),            # every block: twice the bands, the last of three rows
    (13007, 1056, 1152, [27, 35, 19], "6 even bands of 8 rows x 3 rectangles"),   # a band more, rows of different lengths
    (13007, 2112, 992, [18], "11 even bands of 8 rows x 2 rectangles"),           # two more bands of an even number of rows
    (13007, 2112, 1504, [15], "6 even bands of 16 rows x 3 rectangles"),          # bands of 16 rows at most
    (13007, 1504, 1056, [33, 1, 0], "6 bands of 8 rows x 3 rectangles"),          # not even: rows are dealt to the bands by their blocks
    (13007, 2112, 1056, [31] * 16 + [8] * 50, "6 even bands of 16 rows x 3 rectangles"),   # dealt: the longest rows have more than twice the mean
    # dealt: none has, but consecutive rows would make bands of 176 to 264 and 40 blocks where three rectangles have room for 216 (of 47 columns 16 in the largest)
    (13007, 1056, 1504, [44] * 16 + [8] * 17, "6 even bands of 8 rows x 3 rectangles"),
    (13007, 2112, 1056, [22] * 33 + [5] * 33, "6 even bands of 16 rows x 3 rectangles"),
])
def test_even_partitions(cuda, tokens, out_f, in_f, counts, partition):
    dtype = torch.bfloat16
    m = _layer(out_f, in_f, counts, dtype, cuda, 5)
    assert native.matmul_back_kernel_form(tokens, out_f, in_f, m.cols_a.shape[0], dtype).startswith("sdd_bf16_kernel + sdd_reduce_kernel, " + partition)
    print(tokens, out_f, in_f, counts, flush=True)
    g = torch.Generator().manual_seed(tokens)
    x, dy = (torch.randn((tokens, f), generator=g).to(dtype) for f in (in_f, out_f))
    ref = O.matmul_with_output_sparse_support(to64(dy), to64(x), m.build_coo_block_index().cpu().numpy(), (out_f, in_f))
    xd, dyd = x.to(cuda), dy.to(cuda)
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(xd, data, bias, m._buffers, m.schedule()).backward(dyd)
    assert_close(data.grad, ref, dtype, "weight gradient")
    assert_close(bias.grad, to64(dy).sum(0), dtype, "bias gradient")
    assert torch.equal(m.matmul_with_output_sparse_support(dyd, xd), data.grad)   # without the bias gradient
