"""Which bf16 products the column kernel takes by its estimate (the choice is made on the host)."""
import pytest
import torch

from pytorch_block_sparse_amd import native

BF16 = torch.bfloat16


@pytest.mark.parametrize("n, k, tokens, density, transpose, kernel", [
    # faster in the kernel that they have left: 0.87 and 0.91 of its speed in the column kernel
    (1984, 3264, 15459, 0.156, True, "dds16_kernel"),
    (1984, 3200, 16294, 0.166, True, "dds16_kernel"),
    # 0.93 to 0.96: forward products of short contractions with half of the blocks and more
    (2496, 1248, 5380, 0.712, True, "panel_chunk_kernel"),
    (928, 1184, 14262, 0.737, True, "panel_chunk_kernel"),
    # 0.94: input gradients of short contractions at nearly level estimates
    (1408, 1056, 12675, 0.369, False, "panel_chunk_kernel"),
    # of longer ones 1.07 times as fast in the column kernel
    (3936, 2016, 4855, 0.297, False, "ddsc_kernel"),
    # 1.1 to 1.25: the wide kernel's estimate is below the column kernel's bound, but not below the stream kernel's
    (1760, 3232, 10051, 0.19, False, "ddsc_kernel"),
    (2144, 2720, 16379, 0.13, False, "ddsc_kernel"),
    # 1.1 to 1.4 times as fast
    (1728, 2720, 13394, 0.32, True, "ddsc_kernel"),
    (2016, 3936, 15003, 0.0912, True, "ddsc_kernel"),
    (1952, 3072, 13826, 0.1157, False, "ddsc_kernel"),
])
def test_faster_kernel(n, k, tokens, density, transpose, kernel):
    nnz = int(density * (n // 32) * (k // 32))
    assert native.matmul_kernel_name(tokens, n, k, nnz, transpose, BF16) == kernel


@pytest.mark.parametrize("n, k, tokens, per_column, ahead", [
    (4096, 3840, 15649, 35, True),     # 1.07 times as fast
    (3808, 4000, 12795, 47, True),     # 1.05: an odd number of k-blocks
    (3552, 3648, 15579, 44, False),    # level
    (3808, 4000, 12795, 52, False),
    (1376, 3072, 16158, 38, False),    # three groups of columns
    (4096, 3840, 12800, 35, False),    # 98 MB
])
def test_lines_asked_for_ahead(n, k, tokens, per_column, ahead):
    form = native.matmul_kernel_form(tokens, n, k, per_column * (n // 32), False, BF16)
    assert form == ("ddsc_kernel, lines ahead" if ahead else "ddsc_kernel")
