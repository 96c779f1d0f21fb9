"""The fp32 weight gradient of larger problems, on the bf16 matrix cores, against float64: units of one to four blocks, rows without blocks, waves
with few and many chunks, ragged tokens, several slices and launches; its mean error; and what does not fit the bfloat16 parts."""
import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native

pytestmark = pytest.mark.gpu
F32 = torch.float32


def _layer(cuda, out_f, in_f, counts, seed=3):
    rng = np.random.RandomState(seed)
    blocks = [(r, int(c)) for r in range(out_f // 32) for c in rng.choice(in_f // 32, counts[r % len(counts)], replace=False)]
    return BlockSparseMatrix.zeros((out_f, in_f), blocks=blocks, device=cuda)


def _gradients(m, dy, x):
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(m.shape[0], device=x.device, requires_grad=True)
    native.torch_path().linear(x, data, bias, m._buffers, m.schedule()).backward(dy)
    return data.grad, bias.grad


def _want(m, dy, x):
    at = m.build_coo_block_index().long()
    dense = dy.double().t().contiguous() @ x.double()
    return dense.reshape(m.shape[0] // 32, 32, m.shape[1] // 32, 32).permute(0, 2, 3, 1)[at[0], at[1]].reshape(-1, 32)


def _name(m, tokens):
    return native.matmul_back_kernel_name(tokens, m.shape[0], m.shape[1], m.cols_a.shape[0], F32)


@pytest.mark.parametrize("out_f, in_f, tokens, counts", [
    (2048, 2048, 5797, [0, 1, 2, 3, 5, 6, 7, 13, 40, 50]),
    (2048, 2048, 12001, [1, 2, 3, 0, 30]),
    (768, 3072, 9001, [64, 1, 2, 3, 5, 0, 7, 90]),
    (4096, 4096, 700, [128]),      # five or six chunks per wave
    (4096, 4096, 16384, [32]),     # two launches of several slices
])
def test_against_float64(cuda, out_f, in_f, tokens, counts):
    m = _layer(cuda, out_f, in_f, counts)
    print(out_f, in_f, tokens, m.cols_a.shape[0], _name(m, tokens), flush=True)
    assert _name(m, tokens).startswith("sdd_split_kernel")
    torch.manual_seed(tokens)
    x, dy = torch.randn(tokens, in_f, device=cuda), torch.randn(tokens, out_f, device=cuda)
    got, db = _gradients(m, dy, x)
    assert torch.equal(got, m.matmul_with_output_sparse_support(dy, x))   # with the bias gradient: the same sums
    want = _want(m, dy, x)
    off = got.double() - want
    # a wave's chain of chunks of 32 tokens (at most a quarter of all), each chunk with the rounding of a few terms, as in tests/test_gpu_precision.py
    limit = 0.35 * 2.0 ** -24 * np.sqrt(8 + tokens / 128) + 2.0 ** -25
    assert (off.norm() / want.norm()).item() <= limit
    # a rounding that goes one way only would show here: every chunk's error has the same sign then
    assert abs(off.mean().item()) <= 0.1 * limit * want.square().mean().sqrt().item()
    assert ((db.double() - dy.double().sum(0)).norm() / dy.double().sum(0).norm()).item() <= 2e-7


def test_values_that_have_no_parts(cuda):
    m = _layer(cuda, 1024, 1024, [16])
    tokens = 9000
    assert _name(m, tokens).startswith("sdd_split_kernel")
    x, dy = torch.randn(tokens, 1024, device=cuda), torch.randn(tokens, 1024, device=cuda)
    clean = m.matmul_with_output_sparse_support(dy, x)
    coo = m.build_coo_block_index().long()
    x[77, 5], x[8999, 40], dy[4000, 100] = float("inf"), float("nan"), -float("inf")
    got = m.matmul_with_output_sparse_support(dy, x).view(-1, 32, 32)   # [block][input feature][output feature]
    bad = torch.zeros_like(got, dtype=torch.bool)
    bad[coo[1] == 0, 5, :] = True
    bad[coo[1] == 1, 8, :] = True
    bad[coo[0] == 3, :, 4] = True
    assert torch.equal(~torch.isfinite(got), bad)
    assert torch.equal(got[~bad], clean.view(-1, 32, 32)[~bad])
    inf = got[:, 5, :][(coo[1] == 0) & (coo[0] != 3)]
    sign = torch.sign(dy[77].view(32, 32))[coo[0][(coo[1] == 0) & (coo[0] != 3)]]
    assert torch.equal(torch.sign(inf), sign) and torch.isinf(inf).all()
    for scale_x, scale_dy in ((2.0 ** 75, 2.0 ** 20), (2.0 ** -118, 2.0 ** -2), (2.0 ** -60, 2.0 ** -60)):
        x, dy = torch.randn(tokens, 1024, device=cuda) * scale_x, torch.randn(tokens, 1024, device=cuda) * scale_dy
        want = _want(m, dy, x)
        got = m.matmul_with_output_sparse_support(dy, x).double()
        # (the fp32 instructions' chains of a chunk and of a wave's chunks; what products near 2^-120 lose below 2^-149 is far less)
        distance = ((got - want).norm() / want.norm()).item()
        print(scale_x, scale_dy, distance, flush=True)
        assert distance <= 0.35 * 2.0 ** -24 * np.sqrt(32 + tokens / 128) + 2.0 ** -25, (scale_x, scale_dy)


@pytest.mark.parametrize("tokens, counts", [(5797, [26, 27]), (4801, [28])])
def test_bias_gradient_of_long_shares(cuda, tokens, counts):
    """Up to 46 and 38 chunks of a wave one behind the other: what the additions cut off is carried along."""
    m = _layer(cuda, 2048, 2048, counts)
    print(tokens, _name(m, tokens), flush=True)
    assert _name(m, tokens) == "sdd_split_kernel"   # one slice
    torch.manual_seed(tokens)
    x, dy = torch.randn(tokens, 2048, device=cuda), torch.randn(tokens, 2048, device=cuda)
    got, want = _gradients(m, dy, x)[1].double(), dy.double().sum(0)
    # four roundings of a chunk's sum of 16, one of the carried sum, one of two lanes, three of the waves; each at most 2^-24 of what it rounds, a third of that
    # squared on average, in a random walk
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -24 * np.sqrt((4 + 1 + 1 + 3) / 3)
