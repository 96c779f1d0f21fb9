"""The plans that the products derive, as a graph capture and other streams see them.  Results are compared with the same products made eagerly by a second matrix."""
import copy

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix


def _products(m, x, dy):
    return m.reverse_matmul(x, True), m.reverse_matmul(dy, False), m.matmul_with_output_sparse_support(dy, x)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,warm,tokens", [
    (torch.float32, 0, 96),         # nothing derived before the capture
    (torch.bfloat16, 8, 33000),     # other parts of the plans, and rectangles after units
    (torch.bfloat16, 33000, 8),
])
def test_capture_before_the_plans_exist(cuda, dtype, warm, tokens):
    """What a capture derives belongs to its graph: an eager product before the first replay does not rely on it."""
    np.random.seed(7)
    torch.manual_seed(7)
    m = BlockSparseMatrix.randn((512, 2048), 256, device=cuda, dtype=dtype)
    x = torch.randn(max(tokens, 1), 2048, device=cuda).to(dtype)
    dy = torch.randn(max(tokens, 1), 512, device=cuda).to(dtype)
    want = [t.clone() for t in _products(copy.deepcopy(m), x, dy)]   # (also raises the kernels' LDS limits)
    if warm:
        _products(m, torch.randn(warm, 2048, device=cuda).to(dtype), torch.randn(warm, 512, device=cuda).to(dtype))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _products(m, x, dy)
    for _ in range(3):
        for got, ref in zip(_products(m, x, dy), want):
            assert torch.equal(got, ref)
        for t in captured:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(captured, want):
            assert torch.equal(got, ref)


@pytest.mark.gpu
def test_plans_made_on_another_stream(cuda):
    np.random.seed(9)
    torch.manual_seed(9)
    m = BlockSparseMatrix.randn((512, 768), 192, device=cuda)
    x, dy = torch.randn(200, 768, device=cuda), torch.randn(200, 512, device=cuda)
    want = [t.clone() for t in _products(copy.deepcopy(m), x, dy)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    results = []
    for s in streams:   # the first one derives the plans, no other one waits for it
        with torch.cuda.stream(s):
            results.append(_products(m, x, dy))
    torch.cuda.synchronize()
    for got in results:
        for g, w in zip(got, want):
            assert torch.equal(g, w)
