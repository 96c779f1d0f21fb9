"""block_replace and validate_indices of a matrix on the GPU (one kernel each) against the host versions, bit for bit and
message for message: grids whose bitmaps fit LDS and one whose do not, line lengths around multiples of 32."""
import copy

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseLinear, BlockSparseMatrix

pytestmark = pytest.mark.gpu
NAMES = ("blocks", "cols_a", "row_start_ends_a", "rows_b", "col_start_ends_b")


def _pair(X, Y, nnz, cuda):
    np.random.seed(X + Y + nnz)
    host = BlockSparseMatrix.zeros((32 * X, 32 * Y), nnz, device="cpu")
    gpu = BlockSparseMatrix.zeros((32 * X, 32 * Y), nnz, device="cpu").to(cuda)
    gpu.load_state_dict(host.state_dict())
    return host, gpu


@pytest.mark.parametrize("X, Y, nnz, moved", [(1, 2, 1, 1), (31, 33, 200, 20), (64, 32, 1500, 548), (96, 24, 1152, 0), (640, 640, 5000, 1234)])
def test_moves_match_the_host(cuda, X, Y, nnz, moved):
    print(X, Y, nnz, moved, flush=True)
    host, gpu = _pair(X, Y, nnz, cuda)
    for turn in range(2):   # the second turn starts from recycled data blocks
        free = (~host.block_mask_build(None)).nonzero()
        to = free[torch.randperm(free.shape[0])[:moved]]
        rep = torch.cat([to, torch.randperm(nnz)[:moved, None]], 1)
        host.block_replace(rep)
        gpu.block_replace(rep.to(cuda))
        for name in NAMES:
            assert torch.equal(getattr(host, name), getattr(gpu, name).cpu()), name
        gpu.validate_indices()


def test_bad_moves_raise_and_change_nothing(cuda):
    _, gpu = _pair(8, 6, 20, cuda)
    before = {n: getattr(gpu, n).clone() for n in NAMES}
    taken = gpu.build_coo_block_index()[:, 0].tolist()
    for rep in ([[0, 0, 20]], [[0, 0, -1]], [[8, 0, 0]], [[0, -1, 0]], [[taken[0], taken[1], 1]]):
        with pytest.raises(Exception, match="block_replacements"):
            gpu.block_replace(torch.tensor(rep, device=cuda))
        assert all(torch.equal(getattr(gpu, n), before[n]) for n in NAMES)


def test_broken_buffers_give_the_message_of_the_host(cuda):
    host, gpu = _pair(40, 33, 300, cuda)
    ends = host.row_start_ends_a.tolist()
    e0 = next(ends[r] for r in range(40) if ends[r + 1] - ends[r] >= 2)
    nnz = 300
    changes = [("row_start_ends_a", 0, 1), ("row_start_ends_a", 3, nnz + 1), ("row_start_ends_a", 40, nnz + 5), ("col_start_ends_b", 2, -4),
               ("col_start_ends_b", 33, nnz - 1), ("cols_a", (0, 0), 33), ("rows_b", (5, 0), -1), ("cols_a", (7, 1), nnz), ("rows_b", (0, 1), int(host.rows_b[1, 1])),
               ("blocks", 0, 1000), ("blocks", 1, 39 if int(host.blocks[1]) != 39 else 0), ("cols_a", (e0 + 1, 0), int(host.cols_a[e0, 0]))]
    for name, at, value in changes:
        messages = []
        for m in (host, gpu):
            t = getattr(m, name)
            keep = t[at].clone()
            t[at] = value
            with pytest.raises(Exception) as e:
                m.validate_indices()
            messages.append(str(e.value))
            t[at] = keep
            m.validate_indices()
        assert messages[0] == messages[1], (name, at, value)


def _step(layer, x, dy):
    y = layer(x)
    return [y, *torch.autograd.grad(y, (x, layer.weight.get_differentiable_data(), layer.bias), dy)]


def _moves(m, count, seed):
    g = torch.Generator(device=m.blocks.device).manual_seed(seed)
    free = (~m.block_mask_build(None)).nonzero()
    to = free[torch.randperm(free.shape[0], generator=g, device=free.device)[:count]]
    return torch.cat([to, torch.randperm(m.blocks.numel() // 2, generator=g, device=free.device)[:count, None]], 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("other_stream", [False, True])
def test_steps_between_moves_are_those_of_a_fresh_matrix(cuda, dtype, other_stream):
    """A trained matrix has the plans of its new pattern made with the arrays: the same steps as of a copy, which derives its own."""
    np.random.seed(3)
    layer = BlockSparseLinear(416, 1056, density=0.4, device=cuda, dtype=dtype)
    with torch.no_grad():
        layer.weight.data.normal_()
        layer.bias.normal_()
    torch.manual_seed(4)
    x, dy = torch.randn(301, 416, device=cuda).to(dtype).requires_grad_(), torch.randn(301, 1056, device=cuda).to(dtype)
    stream = torch.cuda.Stream() if other_stream else torch.cuda.current_stream()
    for turn in range(4):
        if turn != 1:   # (moves twice without a step between them)
            _step(layer, x, dy)
        moves = _moves(layer.weight, 30 + turn, turn)
        torch.cuda.current_stream().synchronize()
        layer.weight.block_replace(moves)
        with torch.cuda.stream(stream):   # (what block_replace returns is complete for every stream)
            got = _step(layer, x, dy)
            stream.synchronize()
        fresh = copy.deepcopy(layer)
        fresh.weight.validate_indices()
        for a, b in zip(got, _step(fresh, x, dy)):
            assert torch.equal(a, b)


def test_rejected_moves_of_a_trained_matrix(cuda):
    np.random.seed(5)
    layer = BlockSparseLinear(512, 768, density=0.5, device=cuda)
    torch.manual_seed(5)
    x, dy = torch.randn(129, 512, device=cuda, requires_grad=True), torch.randn(129, 768, device=cuda)
    want = _step(layer, x, dy)
    for _ in range(3):
        with pytest.raises(Exception, match="block_replacements"):
            layer.weight.block_replace(torch.tensor([[0, 0, 10 ** 6]], device=cuda))
        assert all(torch.equal(a, b) for a, b in zip(want, _step(layer, x, dy)))


def test_moves_without_room_for_plans(cuda):
    """The moves themselves need a few kilobytes: where the new pattern's plans find no memory, they succeed all the same, and refused ones say why."""
    np.random.seed(7)
    layer = BlockSparseLinear(16384, 16384, density=0.004, device=cuda)   # plans of 2 MB each
    torch.manual_seed(7)
    x, dy = torch.randn(40, 16384, device=cuda, requires_grad=True), torch.randn(40, 16384, device=cuda)
    _step(layer, x, dy)
    layer.weight.block_replace(_moves(layer.weight, 50, 0))
    _step(layer, x, dy)
    moves, bad = _moves(layer.weight, 50, 1), torch.tensor([[0, 0, 10 ** 6]], device=cuda)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total, filler = torch.cuda.get_device_properties(cuda).total_memory, []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while len(filler) < 1 << 16:
                filler.append(torch.empty(3 << 19, dtype=torch.uint8, device=cuda))
        with pytest.raises(Exception, match="block_replacements"):
            layer.weight.block_replace(bad)
        layer.weight.block_replace(moves)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            _step(layer, x, dy)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    filler.clear()
    layer.weight.validate_indices()
    fresh = copy.deepcopy(layer)
    for a, b in zip(_step(layer, x, dy), _step(fresh, x, dy)):
        assert torch.equal(a, b)
