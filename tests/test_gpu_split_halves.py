"""fp32 products on the bf16 cores with columns that two waves share and tiles of 32 tokens: columns of one block to all, next to each other and far apart."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import BlockSparseMatrix, native

pytestmark = pytest.mark.gpu
# blocks per column, of 128: the first ones are heavy (more than twice the average); around the 64 entries that a wave has at hand, and of every length modulo
# the three blocks in flight
UNEVEN = [128, 128, 127, 67, 66, 65, 64, 63, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 1, 3, 2, 0, 1, 4]


@pytest.mark.parametrize("transpose", [True, False])
@pytest.mark.parametrize("tokens, counts", [
    (4096, UNEVEN), (4133, UNEVEN), (8191, UNEVEN), (3300, UNEVEN),   # one group of columns more than without heavy ones
    (4100, [128] * 8 + [9] * 24),                                     # heavy columns alone in their groups
    (4127, [26] * 24),                                                # none: 32-token tiles of sparse columns
])
def test_halves(cuda, tokens, counts, transpose):
    n, k = 32 * len(counts), 4096
    rng = np.random.default_rng(tokens)
    of_column = [np.sort(rng.choice(128, c, replace=False)) if c != 2 else np.array([0, 127]) for c in counts]   # (two: as far apart as can be)
    cells = [(c, int(i)) if transpose else (int(i), c) for c, rows in enumerate(of_column) for i in rows]
    rng.shuffle(cells)
    shape = (n, k) if transpose else (k, n)
    m = BlockSparseMatrix.zeros(shape, blocks=[tuple(int(v) for v in c) for c in cells], device=cuda, dtype=torch.float32)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    with torch.no_grad():
        m.data.normal_(generator=g)
    a = torch.randn((tokens, k), generator=g, device=cuda)
    kernel = native.load().pbs_blocksparse_matmul_kernel_name(tokens, n, k, len(cells), int(transpose), 0, 1)
    assert b"split_kernel" in kernel
    got = m.reverse_matmul(a, transpose=transpose)
    failures = ctypes.c_uint()
    assert native.load().pbs_protocol_failures(ctypes.byref(failures)) == 0 and failures.value == 0
    dense = m.to_dense().double()
    dense = dense.t() if transpose else dense
    rows = torch.cat([torch.arange(0, tokens, 61), torch.arange(tokens - 70, tokens)]).to(cuda)
    want, most = a[rows].double() @ dense.contiguous(), a[rows].double().abs() @ dense.abs().contiguous()
    # a block's twelve products of parts and their sums (32 each) in fp32, the products that are left out, one rounding per block, each 2^-24 of at most the sum of
    # the magnitudes
    bound = (12 * 32 + 1 + max(counts)) * 2.0 ** -24 * most
    assert bool(((got[rows].double() - want).abs() <= bound).all())
    # the bits of a token are the same in any call
    fewer = m.reverse_matmul(a[:tokens - 37].contiguous(), transpose=transpose)
    if b"split_kernel" in native.load().pbs_blocksparse_matmul_kernel_name(tokens - 37, n, k, len(cells), int(transpose), 0, 1):
        assert torch.equal(fewer, got[:tokens - 37])


def test_values_that_have_no_parts(cuda):
    """In both halves of a tile that two waves share, and in a tile of 32 tokens at the end."""
    tokens, k = 8191, 4096
    rng = np.random.default_rng(7)
    m = BlockSparseMatrix.zeros((32 * len(UNEVEN), k), blocks=[(c, int(i)) for c, n in enumerate(UNEVEN) for i in rng.choice(128, n, replace=False)],
                                device=cuda, dtype=torch.float32)
    g = torch.Generator(device="cuda").manual_seed(7)
    with torch.no_grad():
        m.data.normal_(generator=g)
    x = torch.randn((tokens, k), generator=g, device=cuda)
    rows, at = [3, 40, 100, 8170, 8190], [5, 1000, 2000, 3000, 4095]
    x[rows, at] = 0.0
    x[[7, 50, 8180]] *= 2.0 ** 100   # beyond what is scaled
    clean, bad = m.reverse_matmul(x, transpose=True), x.clone()
    bad[rows, at] = torch.tensor([float("inf"), -float("inf"), float("nan"), float("inf"), float("nan")], device=cuda)
    got, w = m.reverse_matmul(bad, transpose=True), m.to_dense()
    reached = torch.zeros_like(got, dtype=torch.bool)
    reached[rows] = (w != 0).t()[at]
    assert reached.any(1)[rows].all() and torch.equal(torch.isfinite(got), ~reached) and torch.equal(got[~reached], clean[~reached])
    want, most = x[[7, 50, 8180]].double() @ w.double().t().contiguous(), x[[7, 50, 8180]].double().abs() @ w.double().t().contiguous().abs()
    # fp32 instructions: a block's chain of 32 products, and one rounding per block
    assert bool(((got[[7, 50, 8180]].double() - want).abs() <= (32 + 1 + max(UNEVEN)) * 2.0 ** -24 * most).all())


@pytest.mark.parametrize("tokens, k, n, nnz, parts", [
    (8192, 1024, 768, 256, True), (8191, 1024, 768, 256, False),   # 2^21 tokens x blocks, and fewer
    (9738, 256, 1184, 168, False), (7337, 960, 448, 246, False), (6317, 640, 2336, 303, False), (1024, 3072, 768, 1600, False),
    (6393, 960, 448, 246, False), (9361, 256, 1184, 168, False),
])
def test_smaller_products(cuda, tokens, k, n, nnz, parts):
    np.random.seed(tokens)
    m = BlockSparseMatrix.randn((n, k), nnz, device=cuda, dtype=torch.float32)
    assert (native.load().pbs_blocksparse_matmul_parts_bytes(tokens, n, k, nnz, 1, 0) > 0) == parts
    g = torch.Generator(device="cuda").manual_seed(tokens)
    a = torch.randn((tokens, k), generator=g, device=cuda)
    got, dense = m.reverse_matmul(a, transpose=True), m.to_dense().double().t().contiguous()
    want, most = a.double() @ dense, a.double().abs() @ dense.abs()
    # as above; with fp32 instructions a chain of at most k products
    assert bool(((got.double() - want).abs() <= max(12 * 32 + 1 + k // 32, k) * 2.0 ** -24 * most).all())
