"""How far the products and gradients are from float64, on inputs without structure.

fp32: a chain of L multiply-adds rounds L times, each time by up to half a unit in the last place of a running sum that grows like
the square root of its length; for a uniform rounding error that makes 0.72 / sqrt(3) / sqrt(2) = 0.29 times 2^-24 sqrt(L) of the
result's size (measured in the products: 0.29 to 0.31).  The bounds below take 0.35 and the chains that the kernels are meant to have: a wave's
share of a column's blocks in the products (2 waves, from 14 blocks per column 4), and in the weight and bias gradient 32 tokens and then the
wave's chunks of 32 tokens, a quarter of all at most.

bf16: sums are float32, so a result is as far from float64 as the rounding of the exact result to bfloat16 is."""
import math

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native
from pytorch_block_sparse_amd.workloads import zipf_positions

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16


def _chain(length):
    return 0.35 * 2.0 ** -24 * math.sqrt(length) + 2.0 ** -25   # and the rounding of what joins the chains


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("out_f, in_f, tokens, blocks", [
    (3072, 768, 4096, 1152), (768, 3072, 101, 1152), (768, 3072, 4096, "zipf"), (256, 1024, 2048, 26), (768, 768, 16384, 288),
    (32, 8736, 70, 273),          # one long column
    (4096, 4096, 2048, 4096), (4096, 4096, 1, 4096),
    (1024, 4096, 16384, 512), (2048, 2048, 16384, 2048), (768, 3072, 2317, 576),
    (2912, 3104, 8117, 8827),     # fp32: the weight gradient in four launches
])
def test_distance_from_float64(cuda, dtype, out_f, in_f, tokens, blocks):
    np.random.seed(1)
    torch.manual_seed(1)
    if blocks == "zipf":
        X, Y = out_f // 32, in_f // 32
        where = [(int(p) // Y, int(p) % Y) for p in zipf_positions(X, Y, X * Y // 4, seed=1)]
        m = BlockSparseMatrix.zeros((out_f, in_f), blocks=where, device=cuda, dtype=dtype)
        m.data.data.normal_()
    else:
        m = BlockSparseMatrix.randn((out_f, in_f), blocks, device=cuda, dtype=dtype)
    nnz = m.cols_a.shape[0]
    print(out_f, in_f, tokens, nnz, dtype, native.matmul_kernel_name(tokens, out_f, in_f, nnz, True, dtype),
          native.matmul_kernel_name(tokens, in_f, out_f, nnz, False, dtype), native.matmul_back_kernel_name(tokens, out_f, in_f, nnz, dtype), flush=True)
    x, dy, bias = (torch.randn(*s, device=cuda).to(dtype) for s in ((tokens, in_f), (tokens, out_f), (out_f,)))
    w = m.to_dense().double()
    at = m.build_coo_block_index().long()
    dense = dy.double().t().contiguous() @ x.double()
    data, b = m.data.detach().clone().requires_grad_(), torch.zeros_like(bias, requires_grad=True)
    native.torch_path().linear(x, data, b, m._buffers, m.schedule()).backward(dy)

    def share(ends, lists):   # blocks of a wave in the fullest column
        return math.ceil(int((ends[1:] - ends[:-1]).max()) / (4 if nnz / lists >= 14.0 else 2))

    of_a_wave = math.ceil(tokens / 128)
    for what, got, want, length in (
        ("forward", m.reverse_matmul(x, True, bias=bias), x.double() @ w.t().contiguous() + bias.double(), 32 * share(m.row_start_ends_a, out_f // 32)),
        ("input gradient", m.reverse_matmul(dy, False), dy.double() @ w, 32 * share(m.col_start_ends_b, in_f // 32)),
        ("weight gradient", data.grad, dense.reshape(out_f // 32, 32, in_f // 32, 32).permute(0, 2, 3, 1)[at[0], at[1]].reshape(-1, 32), 32 + of_a_wave),
        ("bias gradient", b.grad, dy.double().sum(0), 32 + of_a_wave),
    ):
        size = want.norm()
        off = ((got.double() - want).norm() / size).item()
        limit = _chain(length) if dtype == F32 else 1.01 * ((want.to(BF16).double() - want).norm() / size).item()
        print("  %s %.2e of %.2e" % (what, off, limit), flush=True)
        assert off <= limit, what
