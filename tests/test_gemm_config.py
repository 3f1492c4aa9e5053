"""``launch_config`` and the registry's metadata name the GEMM kernel and tile that ``tk_gemm`` picks
(``tk_gemm_tile``): which operands take which kernel, and tiles of every layout. Needs no GPU."""

from __future__ import annotations

import pytest
import torch

from tklab import _hip
from tklab.kernels import matmul
from tklab.registry import REGISTRY


def _matrix(rows: int, cols: int, layout: str, dtype=torch.bfloat16) -> torch.Tensor:
    """An empty matrix: by rows, by columns, by odd rows (no aligned groups) or with no unit stride."""
    if layout == "rows":
        return torch.empty(rows, cols, dtype=dtype)
    if layout == "columns":
        return torch.empty(cols, rows, dtype=dtype).t()
    if layout == "odd":
        return torch.empty(rows, cols + 1, dtype=dtype)[:, 1:]
    if layout == "odd columns":
        return torch.empty(cols, rows + 1, dtype=dtype)[:, 1:].t()
    return torch.empty(rows, 2 * cols, dtype=dtype)[:, ::2]


def _config(m, n, k, a, b):
    config = matmul.launch_config(_matrix(m, k, a), _matrix(k, n, b))
    return config["hip_kernel"], (config["block_m"], config["block_n"]), config["num_stages"]


@pytest.mark.parametrize(("a", "b", "k", "kernel", "stages"), [
    ("rows", "rows", 64, "gemm_dma_kernel", 5), ("rows", "rows", 72, "gemm_kernel", 5),
    ("rows", "columns", 64, "gemm_kernel", 5), ("columns", "rows", 64, "gemm_kernel", 5),
    ("columns", "columns", 64, "gemm_kernel", 5), ("odd", "rows", 64, "gemm_kernel", 2),
    ("rows", "odd columns", 64, "gemm_kernel", 2), ("rows", "strided", 64, "gemm_kernel", 2),
    ("rows", "rows", 63, "gemm_kernel", 2),
])
def test_layouts_take_their_kernel(a, b, k, kernel, stages) -> None:
    assert _config(128, 72, k, a, b) == (kernel, (64, 64), stages)


@pytest.mark.parametrize(("m", "n", "dma", "staged", "strided"), [
    (8, 8, (64, 64), (64, 64), (64, 64)), (416, 4632, (128, 128), (128, 128), (128, 128)),
    (2184, 2728, (256, 128), (256, 128), (128, 128)), (2320, 3680, (256, 256), (256, 128), (128, 128)),
    (824, 4632, (128, 192), (256, 128), (128, 128)),
])
def test_tiles_by_size_and_layout(m, n, dma, staged, strided) -> None:
    """Register-staged tiles are at most 256 x 128; element loads (no unit stride) 128 x 128."""
    k = 416 if (m, n) == (824, 4632) else 96
    assert _config(m, n, k, "rows", "rows")[1] == dma
    assert _config(m, n, k, "odd", "rows")[1] == staged
    assert _config(m, n, k, "strided", "strided")[1] == strided
    # Both transposed: C^T = B^T A^T, the tile of the problem with M and N exchanged.
    assert _config(m, n, k, "columns", "columns")[1] == _config(n, m, k, "rows", "rows")[1]
    assert _config(m, n, k, "odd columns", "odd columns")[1] == _config(n, m, k, "odd", "odd")[1]


def test_registry_sizes_name_the_launchers_kernel() -> None:
    for name in ("matmul_fp32acc", "matmul_fp16acc"):
        spec = REGISTRY[name]
        for size in spec.sizes:
            meta = spec.benchmark_metadata(size, torch.float16)
            square = torch.empty(size, size, dtype=torch.float16)
            assert meta == matmul.launch_config(square, square)


def test_rejected_problems_have_no_tile() -> None:
    for sizes, strides in (((0, 8, 8), (8, 1, 8, 1)), ((8, 8, 8), (0, 1, 8, 1)), ((8, 8, 8), (8, 1, 8, -1)),
                           ((1 << 20, 8, 4096), (4096, 1, 8, 1))):
        assert _hip.query("tk_gemm_tile", 0, 0, *sizes, *strides) == 0
