"""All gradients of a layer in one call: bit for bit those of the separate products, whether or not the launch that adds the weight gradient's slices
also splits the blocks of the input gradient."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseLinear, BlockSparseMatrix, native

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16


def _shared(tokens, in_f, out_f, nnz, dtype):
    """(slices that a launch adds, blocks in parts): with both, one launch does both."""
    lib, code = native.load(), native.DTYPE_CODES[dtype]
    return (lib.pbs_blocksparse_matmul_back_bias_workspace_bytes(tokens, out_f, in_f, nnz, code) > 0,
            lib.pbs_blocksparse_matmul_parts_bytes(tokens, in_f, out_f, nnz, 0, code) > 0)


@pytest.mark.parametrize("dtype, tokens, in_f, out_f, nnz, bias, slices, parts", [
    (F32, 4096, 768, 3072, 1152, True, True, True), (F32, 3072, 3072, 768, 1151, True, True, True), (F32, 4097, 1024, 1024, 1021, False, True, True),
    (F32, 16384, 2048, 2048, 4095, True, True, True),
    (F32, 5797, 2048, 2048, 1696, True, False, True), (F32, 4099, 768, 768, 286, True, True, False), (F32, 130, 768, 3072, 1152, True, False, False),
    (F32, 1, 32, 32, 1, True, False, False), (F32, 64, 416, 160, 0, True, False, False), (F32, 0, 768, 3072, 700, True, False, False),
    (BF16, 2317, 768, 3072, 1152, True, False, False), (BF16, 8192, 2048, 2048, 2000, True, True, False),
])
def test_together_like_apart(cuda, dtype, tokens, in_f, out_f, nnz, bias, slices, parts):
    assert _shared(tokens, in_f, out_f, nnz, dtype) == (slices, parts)
    np.random.seed(nnz)
    layer = BlockSparseLinear(in_f, out_f, bias=bias, density=0.5, device=cuda, dtype=dtype)
    layer.weight = BlockSparseMatrix.randn((out_f, in_f), nnz, device=cuda, dtype=dtype)
    g = torch.Generator(device="cuda").manual_seed(nnz)
    x = torch.randn((tokens, in_f), generator=g, device=cuda, dtype=dtype).requires_grad_(True)
    dy = torch.randn((tokens, out_f), generator=g, device=cuda, dtype=dtype)
    weights = [layer.weight.get_differentiable_data()] + ([layer.bias] if bias else [])
    y = layer(x)
    apart = torch.autograd.grad(y, [x], dy, retain_graph=True) + torch.autograd.grad(y, weights, dy, retain_graph=True)
    together = torch.autograd.grad(y, [x] + weights, dy)
    for a, b in zip(apart, together):
        assert torch.equal(a, b)


def test_workspace_and_arguments(cuda):
    """(Refused before anything is launched: none of these pointers is read.)"""
    lib, p, null = native.load(), ctypes.c_void_p(0x1000), ctypes.c_void_p(0)
    need = lib.pbs_blocksparse_linear_back_workspace_bytes(4096, 3072, 768, 1152, 0)
    assert need >= lib.pbs_blocksparse_matmul_back_bias_workspace_bytes(4096, 3072, 768, 1152, 0) + 1152 * 6144

    def call(dy=p, x=p, data=p, dx=p, units=p, tokens=4096, dtype=0, ws=p, size=need):
        return lib.pbs_blocksparse_linear_back(dy, x, data, p, p, p, units, dx, p, p, tokens, 3072, 768, 1152, dtype, ws, size, null)
    assert call(size=need - 1) == -5 and call(ws=null) == -5 and call(ws=ctypes.c_void_p(0x1008)) == -5
    assert call(dy=null) == -1 and call(x=null) == -1 and call(data=null) == -1 and call(dx=null) == -1 and call(units=null) == -1
    assert call(dx=ctypes.c_void_p(0x1004)) == -4 and call(x=ctypes.c_void_p(0x1004)) == -4
    assert call(x=null, tokens=130) == -1 and call(x=ctypes.c_void_p(0x1004), tokens=130) == -4   # (the input gradient would come first)
    assert call(tokens=-1) == -2 and call(dtype=7) == -3


def test_graph_replays(cuda):
    """A captured step: every replay, with eager steps between them, gives what the eager step gives."""
    np.random.seed(5)
    layer = BlockSparseLinear(3072, 768, density=0.5, device=cuda, dtype=F32)
    assert _shared(4096, 3072, 768, layer.weight.cols_a.shape[0], F32) == (True, True)
    x = torch.randn((4096, 3072), device=cuda).requires_grad_(True)
    dy = torch.randn((4096, 768), device=cuda)
    weights = [layer.weight.get_differentiable_data(), layer.bias]

    def step():
        return torch.autograd.grad(layer(x), [x] + weights, dy)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        with torch.no_grad():
            x.normal_(generator=g)
            dy.normal_(generator=g)
            layer.weight.data.normal_(generator=g)
        eager = step()
        for t in captured:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(captured, eager):
            assert torch.equal(a, b)
