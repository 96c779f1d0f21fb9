"""The memory that the weight gradient asks for: the partial sums of the fp32 kernel stay within 64 MiB however many tokens,
features and blocks there are, because token ranges beyond that are added by further launches."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import block_sparse_oracle as O
from pytorch_block_sparse_amd import native
from tests.helpers import assert_close, to64

MIB = 1 << 20


@pytest.mark.parametrize("out_f, in_f", [(4096, 4096), (8192, 8192), (768, 3072), (12288, 4096), (2048, 2048), (32, 992)])
@pytest.mark.parametrize("density", [0.05, 0.25, 0.5, 1.0])
def test_fp32_partial_sums_are_bounded(out_f, in_f, density):
    lib = native.load()
    nnz = max(1, int(density * (out_f // 32) * (in_f // 32)))
    table = 64 + (nnz // 4 + out_f // 32) * 64
    for tokens in (1, 100, 1024, 4096, 16384, 65536, 1 << 20, 1 << 24):
        assert lib.pbs_blocksparse_matmul_back_workspace_bytes(tokens, out_f, in_f, nnz, 0) <= 64 * MIB + table, tokens
        with_bias = lib.pbs_blocksparse_matmul_back_bias_workspace_bytes(tokens, out_f, in_f, nnz, 0)
        assert with_bias <= 64 * MIB + 24 * 4 * out_f, tokens   # (at most 24 slices)


@pytest.mark.gpu
@pytest.mark.parametrize("out_f, in_f, tokens, blocks", [
    (2912, 3104, 8117, 8827),    # every block: one slice, four launches straight into the result; ragged tokens
    (2912, 3104, 8117, 4300),    # two slices, two launches; rows of any length
    (3008, 3008, 11000, 4200),   # three slices, two launches
    (128, 115008, 1050, 6000),   # two slices, four launches, of which the last has a slice without tokens
])
def test_launches_that_add_up(cuda, out_f, in_f, tokens, blocks):
    lib = native.load()
    rng = np.random.RandomState(blocks)
    mask = np.zeros(out_f // 32 * (in_f // 32), bool)
    mask[rng.choice(mask.size, blocks, replace=False)] = True
    idx = O.build_indices(mask.reshape(out_f // 32, in_f // 32))
    ptr, cols, coo = (torch.from_numpy(a).to(cuda) for a in (idx["row_start_ends_a"], idx["cols_a"], idx["blocks"]))
    torch.manual_seed(blocks)
    x, dy = torch.randn(tokens, in_f, device=cuda), torch.randn(tokens, out_f, device=cuda)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print(out_f, in_f, tokens, blocks, flush=True)
    size = lib.pbs_blocksparse_matmul_back_units_bytes(tokens, out_f, in_f, blocks, 0)
    units = torch.empty(size, dtype=torch.uint8, device=cuda)
    assert lib.pbs_blocksparse_matmul_back_units(p(ptr), p(cols), out_f, in_f, blocks, p(units), size, stream) == 0
    size = lib.pbs_blocksparse_matmul_back_bias_workspace_bytes(tokens, out_f, in_f, blocks, 0)
    ws = torch.full((max(size, 16) // 4,), float("nan"), device=cuda)
    got, db, plain = torch.full((blocks * 32, 32), float("nan"), device=cuda), torch.full((out_f,), float("nan"), device=cuda), None
    for bias in (db, None):   # (the sums do not depend on whether the bias gradient is wanted)
        got.fill_(float("nan"))
        assert lib.pbs_blocksparse_matmul_back_bias(p(dy), p(x), p(ptr), p(cols), p(units), p(got), None if bias is None else p(bias), tokens,
                                                    out_f, in_f, blocks, 0, p(ws), size, stream) == 0
        assert plain is None or torch.equal(plain, got)
        plain = got.clone()
    dense = dy.double().t().contiguous() @ x.double()
    at = coo.view(-1, 2).long()
    want = dense.reshape(out_f // 32, 32, in_f // 32, 32).permute(0, 2, 3, 1)[at[:, 1], at[:, 0]].reshape(-1, 32)
    assert ((got - want).norm() / want.norm()).item() < 2e-7   # as of one launch: partial sums of 32 tokens
    assert_close(db, to64(dy).sum(0), torch.float32, "bias gradient")
    free = torch.full_like(got, float("nan"))
    assert lib.pbs_blocksparse_matmul_back_noalloc(p(dy), p(x), p(ptr), p(cols), p(free), tokens, out_f, in_f, blocks, 0, stream) == 0
    assert ((free - want).norm() / want.norm()).item() < 2e-7
