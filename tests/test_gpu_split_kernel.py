"""Larger fp32 products on the bf16 matrix cores (three bfloat16 parts of every value, six products), against float64, at the sizes where
the kernel's tiles of 64 and 32 tokens, its groups of 8 columns, its lists in windows of 64 and its units per workgroup have an edge; and what
does not fit the parts: infinities, NaN, the ends of the float range."""
import math

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native
from pytorch_block_sparse_amd.workloads import zipf_positions

pytestmark = pytest.mark.gpu
F32 = torch.float32


def _matrix(cuda, out_f, in_f, blocks, seed=1):
    np.random.seed(seed)
    torch.manual_seed(seed)
    if isinstance(blocks, int):
        return BlockSparseMatrix.randn((out_f, in_f), blocks, device=cuda)
    Y = in_f // 32
    m = BlockSparseMatrix.zeros((out_f, in_f), blocks=[(int(p) // Y, int(p) % Y) for p in blocks], device=cuda)
    m.data.data.normal_()
    return m


def _kernel(m, tokens, transpose):
    n, k = m.shape if transpose else m.shape[::-1]
    return native.matmul_kernel_name(tokens, n, k, m.cols_a.shape[0], transpose, F32)


def _distance(m, x, got, transpose, bias=None):
    w = m.to_dense().double()
    w = w.t().contiguous() if transpose else w
    off = size = 0.0
    for lo in range(0, x.shape[0], 65536):
        want = x[lo:lo + 65536].double() @ w
        if bias is not None:
            want += bias.double()
        off += (got[lo:lo + 65536].double() - want).square().sum().item()
        size += want.square().sum().item()
    return math.sqrt(off / size)


def _fullest(m, transpose):
    ends = m.row_start_ends_a if transpose else m.col_start_ends_b
    return int((ends[1:] - ends[:-1]).max())


def _limit(m, transpose):
    """A rounding for each block of the fullest column, of a sum that grows as those of tests/test_gpu_precision.py do, and those of the blocks' own
    sums and of the result."""
    return 0.35 * 2.0 ** -24 * math.sqrt(_fullest(m, transpose)) + 2.0 ** -25


CASES = [
    (3072, 768, 4096, 1152),       # three full rounds of units
    (768, 3072, 2317, 1152),       # low tiles, the last one ragged
    (1632, 1024, 1501, 1468),      # 51 columns: waves without a column
    (256, 4384, 4701, 1000),       # lists over two windows
    (2048, 65536, 2017, 26300),    # the longest contraction
    (4096, 4096, 512, 4096),       # low tiles alone
    (256, 32, 1040039, 8),         # one k-block, more units than the heads of one workgroup hold
    (768, 3072, 4096, zipf_positions(24, 96, 576, seed=3)),
    (928, 3072, 5061, zipf_positions(29, 96, 900, seed=4)),   # columns of two waves in a group more, low tiles
    (2560, 1600, 1300, [r * 50 + c for r in range(80) for c in range(50) if r < 30 or (r + c) % 10 == 0]),   # as many of them as there can be
    (768, 3072, 4096, [r * 96 + c for r in range(24) for c in range(96) if r % 3 and (r + c) % 2]),   # every third column empty
]


@pytest.mark.parametrize("out_f, in_f, tokens, blocks", CASES)
def test_against_float64(cuda, out_f, in_f, tokens, blocks):
    m = _matrix(cuda, out_f, in_f, blocks)
    bias = torch.randn(out_f + 1, device=cuda)[1:]   # aligned to four bytes
    for transpose in (True, False):
        name = _kernel(m, tokens, transpose)
        print(out_f, in_f, tokens, m.cols_a.shape[0], transpose, name, flush=True)
        if transpose:
            assert name == "split_kernel"
        x = torch.randn(tokens, in_f if transpose else out_f, device=cuda)
        b = bias.clone() if transpose else None
        got = m.reverse_matmul(x, transpose, bias=b)
        assert _distance(m, x, got, transpose, b) <= (_limit(m, transpose) if name == "split_kernel" else 1e-6)
        if b is not None:   # the same bits with a bias anywhere
            plan = native.blocksparse_matmul_plan(m.row_start_ends_a, m.cols_a, out_f, in_f)
            assert torch.equal(native.blocksparse_matmul(x, m.data.detach(), plan, out_f, in_f, m.cols_a.shape[0], True, bias=bias), got)


@pytest.mark.parametrize("out_f, in_f, blocks", [(3072, 768, 1152), (768, 3072, 1152), (1024, 1024, 512), (4096, 4096, 12288)])
def test_sums_of_one_sign_and_their_mean_error(cuda, out_f, in_f, blocks):
    """A chain of roundings over a whole column is further off than the fp32 instructions' where the terms do not cancel, and roundings that go one way
    only show in the mean."""
    m = _matrix(cuda, out_f, in_f, blocks)
    tokens = 4096
    assert _kernel(m, tokens, True) == "split_kernel"
    x = torch.randn(tokens, in_f, device=cuda)
    w = m.to_dense().double().t().contiguous()
    off, size = m.reverse_matmul(x, True).double() - x.double() @ w, (x.double() @ w).square().mean().sqrt()
    print(off.mean().item() / size.item(), flush=True)
    assert abs(off.mean()) <= 0.05 * _limit(m, True) * size
    m.data.data.uniform_()
    x.uniform_()
    for sign in (1.0, -1.0):
        # the sum grows with the blocks: a rounding of it is sqrt(2 / 3) of that above on average
        assert _distance(m, x * sign, m.reverse_matmul(x * sign, True), True) <= _limit(m, True) * math.sqrt(2 / 3)


def test_result_of_a_token_does_not_depend_on_the_others(cuda):
    m = _matrix(cuda, 768, 3072, 1152)
    x = torch.randn(16384, 3072, device=cuda)
    y = m.reverse_matmul(x, True)
    for lo, hi in ((0, 2048), (77, 2394), (33, 9000)):
        assert _kernel(m, hi - lo, True) == "split_kernel"
        assert torch.equal(m.reverse_matmul(x[lo:hi], True), y[lo:hi])
    x[5, 7], x[700, 1] = float("inf"), float("nan")
    ok = torch.ones(16384, dtype=torch.bool, device=cuda)
    ok[5] = ok[700] = False
    assert torch.equal(m.reverse_matmul(x, True)[ok], y[ok])


@pytest.mark.parametrize("transpose", [True, False])
def test_values_that_have_no_parts(cuda, transpose):
    """Where the fp32 instructions give a number the parts have to, and the other way round."""
    m = _matrix(cuda, 1024, 1024, 512)
    tokens = 4200
    assert _kernel(m, tokens, transpose) == "split_kernel"
    w = m.to_dense().double()
    w = w.t().contiguous() if transpose else w
    x = torch.randn(tokens, 1024, device=cuda)
    x[3, 40], x[64, 9], x[65, 8] = float("inf"), float("nan"), -float("inf")
    x[100] *= 2.0 ** 100            # beyond what is scaled
    x[101] *= 2.0 ** -118           # the third parts would be denormal
    x[102] *= 2.0 ** -126
    x[103] = 0.0
    got = m.reverse_matmul(x, transpose)
    present = (w != 0).double()
    for row, value in ((3, 40), (64, 9), (65, 8)):
        reached = present[value] > 0
        assert torch.equal(torch.isfinite(got[row]), ~reached)
    assert torch.equal(torch.sign(got[3])[present[40] > 0], torch.sign(w[40])[present[40] > 0].float())
    assert (got[103] == 0).all()
    for row in (100, 101, 102):
        want = x[row].double() @ w
        # (again with fp32 instructions: 32 roundings of a block's sum and one for each block; of denormal products they keep what is above 2^-149)
        limit = 0.35 * 2.0 ** -24 * math.sqrt(32 + _fullest(m, transpose)) + 2.0 ** -25 if row == 100 else 1e-6
        distance = ((got[row].double() - want).norm() / want.norm()).item()
        print(row, distance, limit, flush=True)
        assert distance <= limit, row
    rest = torch.ones(tokens, dtype=torch.bool, device=cuda)
    rest[[3, 64, 65, 100, 101, 102, 103]] = False
    assert _distance(m, x[rest], got[rest], transpose) <= _limit(m, transpose)
    m.data.data[70, 3] = float("inf")   # (block 2)
    r, c = int(m.blocks[5]), int(m.blocks[4])
    n, k = (32 * r + 3, 32 * c + 6) if transpose else (32 * c + 6, 32 * r + 3)
    got = m.reverse_matmul(x[200:], transpose)
    bad = ~torch.isfinite(got)
    assert bad[:, n].all() and bad.sum() == got.shape[0]
    assert torch.equal(torch.sign(got[:, n]), torch.sign(x[200:, k]))


def test_graph_replays(cuda):
    m = _matrix(cuda, 768, 768, 288)
    x = torch.randn(8000, 768, device=cuda)
    assert _kernel(m, 8000, True) == "split_kernel"
    want = m.reverse_matmul(x, True).clone(), m.reverse_matmul(x, False).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m.reverse_matmul(x, True), m.reverse_matmul(x, False)
    for _ in range(3):
        for o, w in zip(out, want):
            assert torch.equal(m.reverse_matmul(x, w is want[0]), w)
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for o, w in zip(out, want):
            assert torch.equal(o, w)
