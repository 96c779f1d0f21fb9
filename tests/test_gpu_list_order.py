"""Index lists that no host layer has looked at, through the C ABI: entries in any order, entries outside the range and several
entries of one position give the product of the entries that are left, by position, to the last bit."""
import ctypes

import numpy as np
import pytest
import torch

from pytorch_block_sparse_amd import native

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16


def _lists(n, k, per_column, repeats, seed):
    """(dirty, clean) as (ptr, entries [nnz, 2]): the clean list holds the first good entry of every k-block, sorted."""
    rng = np.random.RandomState(seed)
    cols, kb = n // 32, k // 32
    nnz = cols * per_column
    ids = rng.permutation(nnz)
    dirty, clean, ends = [], [], [0]
    for c in range(cols):
        mine = [[int(x), int(ids[c * per_column + i])] for i, x in enumerate(rng.permutation(kb)[:per_column])]
        if c % 3 == 0:
            for at, bad in ((0, [-1, mine[0][1]]), (len(mine) // 2, [kb + 5, mine[1][1]]), (2, [mine[2][0], nnz + 7]), (1, [mine[3][0], -3])):
                mine[at] = bad
        if repeats and c % 4 == 1:
            mine[-1] = [mine[0][0], mine[-1][1]]
        first = {}
        for x, b in mine:
            if 0 <= x < kb and 0 <= b < nnz:
                first.setdefault(x, b)
        dirty += mine
        clean += sorted(first.items())
        ends.append(len(clean))
    clean += [(0, 0)] * (nnz - len(clean))   # (past the last list)
    starts = np.arange(0, nnz + 1, per_column)
    return (starts, np.array(dirty)), (np.array(ends), np.array(clean))


@pytest.mark.parametrize("kernel, dtype, n, k, tokens, per_column, transpose", [
    ("stream_kernel", F32, 256, 1024, 70, 20, True),
    ("stream_kernel", F32, 96, 6400, 33, 130, False),       # more than 64 entries per wave
    ("stream_kernel", BF16, 320, 768, 40, 12, True),
    ("panel_kernel", BF16, 3072, 768, 2317, 12, True),
    ("panel_kernel", BF16, 2048, 768, 8229, 24, False),     # full columns
    ("panel_chunk_kernel", BF16, 768, 3072, 2317, 48, True),
    ("panel_chunk_kernel", BF16, 2048, 2048, 4093, 13, False),
    ("dds16_kernel", BF16, 1024, 4096, 16384, 16, False),
])
def test_products(cuda, kernel, dtype, n, k, tokens, per_column, transpose):
    lib = native.load()
    nnz = n // 32 * per_column
    name = native.matmul_kernel_name(tokens, n, k, nnz, transpose, dtype, False)
    print(name, dtype, n, k, tokens, per_column, flush=True)
    assert name == kernel
    torch.manual_seed(n)
    a, data = torch.randn(tokens, k, device=cuda).to(dtype), torch.randn(nnz * 32, 32, device=cuda).to(dtype)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for ptr, entries in _lists(n, k, per_column, kernel != "dds16_kernel", 7):
        ptr, entries = (torch.from_numpy(x.astype(np.int32)).to(cuda) for x in (ptr, entries))
        plan = native.blocksparse_matmul_plan(ptr, entries, n, k)
        y = torch.full((tokens, n), float("nan"), dtype=dtype, device=cuda)
        assert lib.pbs_blocksparse_matmul(p(a), p(data), p(plan), None, p(y), tokens, n, k, nnz, int(transpose), native.DTYPE_CODES[dtype], stream) == 0
        out.append(y)
    assert torch.isfinite(out[1]).all() and torch.equal(*out)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_weight_gradient_of_entries_outside_the_range(cuda, dtype):
    """They get no result, the others theirs."""
    lib = native.load()
    out_f, in_f, tokens, per_row = 256, 1024, 70, 20
    (ptr, entries), _ = _lists(out_f, in_f, per_row, False, 9)
    nnz = len(entries)
    torch.manual_seed(1)
    x, dy = torch.randn(tokens, in_f, device=cuda).to(dtype), torch.randn(tokens, out_f, device=cuda).to(dtype)
    got = torch.full((nnz, 32, 32), 7.0, dtype=dtype, device=cuda)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    dptr, dent = (torch.from_numpy(v.astype(np.int32)).to(cuda) for v in (ptr, entries))
    code = native.DTYPE_CODES[dtype]
    size = lib.pbs_blocksparse_matmul_back_workspace_bytes(tokens, out_f, in_f, nnz, code)
    ws = torch.empty(max(size, 16), dtype=torch.uint8, device=cuda)
    assert lib.pbs_blocksparse_matmul_back(p(dy), p(x), p(dptr), p(dent), p(got), tokens, out_f, in_f, nnz, code, p(ws), size,
                                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    want = torch.full((nnz, 32, 32), 7.0, dtype=torch.float64)
    for e, (c, b) in enumerate(entries):
        if 0 <= c < in_f // 32 and 0 <= b < nnz:
            r = e // per_row
            want[b] = x[:, 32 * c:32 * c + 32].double().cpu().t() @ dy[:, 32 * r:32 * r + 32].double().cpu()
    assert (got.double().cpu() - want).norm() / want.norm() < (1e-5 if dtype == F32 else 1e-2)


def _split_product(a, data, ptr, entries, n, k, transpose):
    """The product through the entry that takes a workspace, with a plan in memory that holds something else where no list has an entry."""
    lib, cuda = native.load(), a.device
    tokens, nnz = a.shape[0], len(entries)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr, entries = (torch.from_numpy(np.asarray(v).astype(np.int32)).to(cuda) for v in (ptr, entries))
    plan = torch.full((lib.pbs_blocksparse_matmul_plan_part_bytes(n, k),), 0x7f, dtype=torch.uint8, device=cuda)
    assert lib.pbs_blocksparse_matmul_plan_part(p(ptr), p(entries), n, k, nnz, 1, p(plan), plan.numel(), stream) == 0
    code = native.DTYPE_CODES[F32]
    size = lib.pbs_blocksparse_matmul_parts_bytes(tokens, n, k, nnz, int(transpose), code)
    name = native.matmul_kernel_name(tokens, n, k, nnz, transpose, F32, True)
    print(name, n, k, tokens, nnz, transpose, flush=True)
    assert name == "split_kernel" and size > 0
    ws = torch.empty(size, dtype=torch.uint8, device=cuda)
    y = torch.full((tokens, n), float("nan"), device=cuda)
    assert lib.pbs_blocksparse_matmul_ws(p(a), p(data), p(plan), None, p(y), tokens, n, k, nnz, int(transpose), code, p(ws), size, stream) == 0
    return y


@pytest.mark.parametrize("n, k, tokens, per_column, transpose", [(768, 3072, 4096, 48, True), (2048, 4384, 1100, 70, False)])
def test_larger_fp32_products(cuda, n, k, tokens, per_column, transpose):
    torch.manual_seed(n)
    a, data = torch.randn(tokens, k, device=cuda), torch.randn(n // 32 * per_column * 32, 32, device=cuda)
    out = [_split_product(a, data, ptr, entries, n, k, transpose) for ptr, entries in _lists(n, k, per_column, True, 7)]
    assert torch.isfinite(out[1]).all() and torch.equal(*out)


@pytest.mark.parametrize("first, counts", [
    (1152, [0] * 24),                # no entries
    (0, [0] * 24),
    (1104, [0] * 23 + [48]),         # the last column's alone
    (576, [0] * 12 + [48] * 12),
    (336, [0, 48, 0] * 8),
    (3, [90, 0, 0, 1, 0, 0, 0, 2, 0, 64, 65, 0] * 2),
])
def test_larger_fp32_products_of_short_lists(cuda, first, counts):
    """Pointer arrays that start above 0 leave entries of the plan unwritten: columns without entries must not read one."""
    n, k, tokens, nnz = 768, 3072, 4096, 1152
    rng = np.random.RandomState(3)
    ptr = np.cumsum([first] + counts)
    entries = np.zeros((nnz, 2), dtype=np.int64)
    entries[first:ptr[-1], 1] = rng.permutation(nnz)[:sum(counts)]
    for c, count in enumerate(counts):
        entries[ptr[c]:ptr[c + 1], 0] = np.sort(rng.permutation(k // 32)[:count])
    torch.manual_seed(1)
    a, data = torch.randn(tokens, k, device=cuda), torch.randn(nnz * 32, 32, device=cuda)
    got = _split_product(a, data, ptr, entries, n, k, True)
    want = torch.zeros(tokens, n, dtype=torch.float64, device=cuda)
    for c in range(n // 32):
        for x, b in entries[ptr[c]:ptr[c + 1]]:
            want[:, 32 * c:32 * c + 32] += a[:, 32 * x:32 * x + 32].double() @ data[32 * b:32 * b + 32].double()
    # as in tests/test_gpu_split_kernel.py: four roundings per block of the fullest column, and that of the result
    limit = 0.35 * 2.0 ** -24 * (4 * max(counts)) ** 0.5 + 2.0 ** -25
    assert (got.double() - want).norm() <= limit * want.norm()


def test_lists_of_anything(cuda):
    """Every other column has all entries, in any order, many to a k-block: the first good one of each is found in about the time that the entries take to read."""
    n, k, nnz = 512 * 32, 512 * 32, 100000
    lib, rng = native.load(), np.random.RandomState(2)
    ptr = np.array([0, nnz] * 256 + [0])
    entries = np.stack([rng.randint(-3, 515, nnz), rng.randint(-5, nnz + 5, nnz)], 1)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    dptr, dent = (torch.from_numpy(v.astype(np.int32)).to(cuda) for v in (ptr, entries))
    plan = torch.full((lib.pbs_blocksparse_matmul_plan_part_bytes(n, k),), 0x7f, dtype=torch.uint8, device=cuda)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    times = []
    for _ in range(3):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        assert lib.pbs_blocksparse_matmul_plan_part(p(dptr), p(dent), n, k, nnz, 1, p(plan), plan.numel(), stream) == 0
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    print(times, flush=True)
    first = {}
    for x, b in entries:
        if 0 <= x < 512 and 0 <= b < nnz:
            first.setdefault(int(x), int(b))
    want = np.array(sorted(first.items()))
    records = plan.view(torch.int32).cpu().numpy()[:512 * 514 * 2].reshape(512, 514, 2)
    assert [tuple(r[0]) for r in records] == [(c, len(want)) for c in range(0, 512, 2)] + [(c, 0) for c in range(1, 512, 2)]
    for r in records[:256]:
        assert np.array_equal(r[2:2 + len(want)], want)
    assert min(times) < 5.0   # ms; 100000 entries of a wave are three times 1563 loads
