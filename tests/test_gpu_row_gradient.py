"""The weight-gradient kernel with up to four blocks of a block row per workgroup, and the bias gradient that comes with it,
against float64: token counts around the 32-token chunk, rows of 0 to 13 blocks, more block rows than the table kernel keeps in
LDS, one and several token slices."""
import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import BlockSparseMatrix, native
from tests.helpers import assert_close, to64

pytestmark = pytest.mark.gpu
ROWS = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13]   # blocks of a block row


def _layer(out_f, in_f, counts, dtype, device, seed):
    rng = np.random.RandomState(seed)
    blocks = [(r, int(c)) for r in range(out_f // 32) for c in rng.choice(in_f // 32, counts[r % len(counts)], replace=False)]
    return BlockSparseMatrix.zeros((out_f, in_f), blocks=blocks, device=device, dtype=dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,out_f,in_f,counts,slices", [
    (1, 384, 416, ROWS, False), (31, 384, 416, ROWS, False), (32, 384, 416, ROWS, False), (33, 384, 416, ROWS, False),
    (97, 384, 416, ROWS, False), (160, 384, 416, ROWS, False), (161, 384, 416, [13], False), (2317, 384, 416, ROWS, True),
    (4096, 32, 64, [2], True), (16415, 64, 32, [0, 1], True), (45, 32 * 1030, 64, [2, 0, 1], False),
])
def test_row_kernel(cuda, dtype, tokens, out_f, in_f, counts, slices):
    m = _layer(out_f, in_f, counts, dtype, cuda, 3)
    nnz = m.cols_a.shape[0]
    name = native.matmul_back_kernel_name(tokens, out_f, in_f, nnz, dtype)
    print(name, tokens, out_f, in_f, nnz, dtype, flush=True)
    assert name.startswith("sdd_row_kernel") and name.endswith("sdd_reduce_kernel") == slices, name
    g = torch.Generator().manual_seed(tokens)
    x, dy = (torch.randn((tokens, f), generator=g).to(dtype) for f in (in_f, out_f))
    coo = m.build_coo_block_index().cpu().numpy()
    ref = O.matmul_with_output_sparse_support(to64(dy), to64(x), coo, (out_f, in_f))
    xd, dyd = x.to(cuda), dy.to(cuda)
    got = m.matmul_with_output_sparse_support(dyd, xd)
    assert_close(got, ref, dtype, "weight gradient")

    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(xd, data, bias, m._buffers, m.schedule()).backward(dyd)
    assert torch.equal(data.grad, got)   # with the bias gradient: the same sums
    assert_close(bias.grad, to64(dy).sum(0), dtype, "bias gradient")


def _followed_by_nan(shape, dtype, device, seed):
    """A tensor whose memory goes on with NaN behind its last row."""
    g = torch.Generator(device=device).manual_seed(seed)
    whole = torch.full((shape[0] + 64, shape[1]), float("nan"), dtype=dtype, device=device)
    whole[:shape[0]] = torch.randn(shape, generator=g, device=device).to(dtype)
    return whole[:shape[0]]


@pytest.mark.parametrize("dtype, out_f, in_f, counts, kernel", [
    (torch.float32, 384, 416, ROWS, "sdd_row_kernel"), (torch.bfloat16, 384, 416, ROWS, "sdd_row_kernel"),
    (torch.float32, 4096, 4096, [60, 61, 62, 63], "sdd_split_kernel"),
])
@pytest.mark.parametrize("past", [1, 7, 8, 9, 15, 16, 17, 24, 31])
def test_last_chunk_ends_with_the_matrix(cuda, dtype, out_f, in_f, counts, kernel, past):
    """Tokens behind the last one count as zeros, whatever the memory there holds; a copy instruction covers 8 (fp32) or 16 (bf16) of a chunk's 32."""
    tokens = (4096 if kernel == "sdd_split_kernel" else 96) + past
    m = _layer(out_f, in_f, counts, dtype, cuda, past)
    name = native.matmul_back_kernel_name(tokens, out_f, in_f, m.cols_a.shape[0], dtype)
    print(name, tokens, out_f, in_f, dtype, flush=True)
    assert name.startswith(kernel)
    x, dy = _followed_by_nan((tokens, in_f), dtype, cuda, 1), _followed_by_nan((tokens, out_f), dtype, cuda, 2)
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(x, data, bias, m._buffers, m.schedule()).backward(dy)
    at = m.build_coo_block_index().long()
    dense = dy.double().t().contiguous() @ x.double()
    want = dense.reshape(out_f // 32, 32, in_f // 32, 32).permute(0, 2, 3, 1)[at[0], at[1]].reshape(-1, 32)
    # (rtol of the oracle comparisons above; bf16: half a unit of the result)
    limit = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    assert (data.grad.double() - want).norm() <= limit * want.norm()
    assert (bias.grad.double() - dy.double().sum(0)).norm() <= limit * dy.double().sum(0).norm()


@pytest.mark.parametrize("tokens, out_f, counts, kernel", [
    (32, 384, [2], "sdd_row_kernel"), (64, 384, [2], "sdd_row_kernel"),   # one chunk a wave
    (257, 384, ROWS, "sdd_row_kernel"), (500, 384, [0, 2], "sdd_row_kernel"), (2317, 384, [0, 1], "sdd_row_kernel + sdd_reduce_kernel"),
    (2200, 1024, [40, 0, 38], "sdd_split_kernel"), (4103, 384, [60, 0, 63], "sdd_split_kernel + sdd_reduce_kernel"),
])
def test_bias_gradient_of_infinities(cuda, tokens, out_f, counts, kernel):
    """An infinity, a sum that overflows and NaN come out as they do of a plain sum, whichever chunk of a wave's share they are in, in rows with and
    without blocks."""
    in_f = 2048
    m = _layer(out_f, in_f, counts, torch.float32, cuda, 5)
    nnz = m.cols_a.shape[0]
    print(kernel, tokens, out_f, nnz, flush=True)
    assert native.matmul_back_kernel_name(tokens, out_f, in_f, nnz, torch.float32) == kernel
    inf, nan, big = float("inf"), float("nan"), 2.0 ** 127
    torch.manual_seed(tokens)
    dy = torch.randn(tokens, out_f, device=cuda)
    x = torch.randn(tokens, in_f, device=cuda)
    want = {0: inf, 1: -inf, 2: nan, 3: nan, 4: inf, 5: -inf}
    for at in (0, tokens // 2, tokens - 1):   # the first chunk, one in between and the last
        here, other = dy.clone(), (at + 128) % tokens   # (the next chunk of the same wave, if there is one)
        for row in range(out_f // 32):
            f = 32 * row
            here[at, f], here[at, f + 1], here[at, f + 2] = inf, -inf, nan
            here[at, f + 3], here[other, f + 3] = inf, -inf
            here[:, f + 4:f + 6] = 0.0
            here[at, f + 4], here[other, f + 4] = big, big
            here[at, f + 5], here[other, f + 5] = -big, -big
        if other == at:
            here[at, 3::32], here[at, 4::32], here[at, 5::32] = nan, inf, -inf
        data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, device=cuda, requires_grad=True)
        native.torch_path().linear(x, data, bias, m._buffers, m.schedule()).backward(here)
        got = bias.grad.view(-1, 32)
        for i, value in want.items():
            assert torch.equal(got[:, i], torch.full_like(got[:, i], value)) or (value != value and bool(got[:, i].isnan().all())), (at, i, got[:, i].tolist())
        rest = here.double().sum(0).view(-1, 32)[:, 6:]
        # (a chunk's sums in three levels, the four waves and the slices: fewer than 16 roundings of 2^-24)
        assert bool(((got[:, 6:].double() - rest).abs() <= 16 * 2.0 ** -24 * here.double().abs().sum(0).view(-1, 32)[:, 6:]).all())


def _wide_rows(cuda, dtype, out_f, tokens):
    rows = [0, 5, out_f // 64, out_f // 32 - 1]
    m = BlockSparseMatrix.zeros((out_f, 64), blocks=[(r, r % 2) for r in rows], device=cuda, dtype=dtype)
    dy = torch.zeros(tokens, out_f, dtype=dtype, device=cuda)
    torch.manual_seed(2)
    x = torch.randn(tokens, 64, device=cuda).to(dtype)
    for r in rows:
        dy[:, 32 * r:32 * r + 32] = torch.randn(tokens, 32, device=cuda).to(dtype)
    print(dtype, out_f, flush=True)
    got = m.matmul_with_output_sparse_support(dy, x).double()
    at = m.build_coo_block_index().tolist()
    want = torch.cat([x[:, 32 * c:32 * c + 32].double().t().contiguous() @ dy[:, 32 * r:32 * r + 32].double() for r, c in zip(*at)])
    assert (got - want).norm() <= (1e-6 if dtype == torch.float32 else 2.0 ** -8) * want.norm()


@pytest.mark.parametrize("dtype, out_f", [(torch.float32, 1 << 25), (torch.bfloat16, 1 << 26)])
def test_chunks_of_four_gigabytes(cuda, dtype, out_f):
    """A chunk of 32 tokens that is too large to be addressed as one buffer."""
    _wide_rows(cuda, dtype, out_f, 45)


@pytest.mark.parametrize("dtype, out_f, tokens", [(torch.float32, 1 << 27, 33), (torch.bfloat16, 1 << 27, 45), (torch.bfloat16, 1 << 28, 33), (torch.float32, 1 << 28, 17)])
def test_rows_of_half_a_gigabyte(cuda, dtype, out_f, tokens):
    """The rows that one copy instruction reads, 8 (fp32) or 16, have 4 GB and more."""
    _wide_rows(cuda, dtype, out_f, tokens)


@pytest.mark.parametrize("tokens,out_f,in_f,counts", [
    (16391, 1600, 512, [7, 0, 3, 16]),     # one rectangle per band sums all 16 rows; the last band has two
    (17000, 1024, 544, [9, 1]),            # two rectangles share the rows, the second with a single column
    (13007, 1056, 1056, [30, 2, 2, 2]),    # uneven rows are dealt to the bands; three rectangles: 6, 6 and 4 rows
    (2600, 64, 10240, [90]),               # more rectangles than rows
    (16384, 1024, 1024, [0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 2]),   # rectangles without blocks
])
def test_bias_gradient_of_rectangles(cuda, tokens, out_f, in_f, counts):
    dtype = torch.bfloat16
    m = _layer(out_f, in_f, counts, dtype, cuda, 7)
    name = native.matmul_back_kernel_name(tokens, out_f, in_f, m.cols_a.shape[0], dtype)
    print(name, tokens, out_f, in_f, flush=True)
    assert name.startswith("sdd_bf16_kernel")
    g = torch.Generator().manual_seed(tokens)
    x, dy = (torch.randn((tokens, f), generator=g).to(dtype).to(cuda) for f in (in_f, out_f))
    data, bias = m.data.detach().clone().requires_grad_(), torch.zeros(out_f, dtype=dtype, device=cuda, requires_grad=True)
    native.torch_path().linear(x, data, bias, m._buffers, m.schedule()).backward(dy)
    assert_close(bias.grad, to64(dy).sum(0), dtype, "bias gradient")
    assert torch.equal(data.grad, m.matmul_with_output_sparse_support(dy, x))   # (checked against the oracle without it)


def test_fp32_sums_stay_close_to_float64(cuda):
    """768 -> 768, 16384 tokens: each partial sum covers 32 tokens, so the error does not grow with the length of a wave's share.
    A random walk of 32 roundings of 2^-24 gives about 2e-7 of a sum's size; one chain over a wave's share gave 4e-7."""
    m = _layer(768, 768, [12], torch.float32, cuda, 3)
    torch.manual_seed(3)
    x, dy = torch.randn(16384, 768, device=cuda), torch.randn(16384, 768, device=cuda)
    got = m.matmul_with_output_sparse_support(dy, x).double()
    coo = m.build_coo_block_index().long()
    dense = dy.double().t().contiguous() @ x.double()
    want = dense.reshape(24, 32, 24, 32).permute(0, 2, 3, 1)[coo[0], coo[1]].reshape(-1, 32)
    assert ((got - want).norm() / want.norm()).item() < 2e-7
