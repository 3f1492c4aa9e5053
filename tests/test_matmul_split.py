"""Split-K GEMM (``tk_gemm_splitk``): runs of K summed in order of K by a second kernel."""

from __future__ import annotations

import pytest
import torch

from tklab import _hip
from tklab.kernels import matmul, matmul_swiglu, rms_norm_matmul, swiglu


@pytest.mark.parametrize(("m", "n", "k"), [(1, 8, 64), (64, 64, 2048), (16, 4096, 4096), (65, 2000, 8192),
                                           (1024, 1024, 1024), (8192, 8192, 8192), (64, 64, 1 << 20)])
def test_split_rule_leaves_no_run_empty(m: int, n: int, k: int) -> None:
    """At least sixteen 64-wide K tiles a run, symmetric in M and N (C^T = B^T A^T splits alike)."""
    splits = matmul.split_k(m, n, k)
    assert 1 <= splits <= max(1, -(-k // 64) // 16)
    assert splits == matmul.split_k(n, m, k)
    assert splits == 1 or splits * -(-m // 64) * -(-n // 64) <= 256


def _split(a, b, splits, *, up=None, row_scale=None):
    out = torch.empty((a.shape[0], b.shape[1]), device=a.device, dtype=a.dtype)
    matmul.enqueue_split(a, b, out, splits, up=up, row_scale=row_scale)
    return out


# K of whole tiles, one chunk past, one short; N of one lane group, not a multiple of four
# (transposed operands only), one past a tile; more runs than divide the K tiles.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize(("m", "n", "k", "splits"), [(8, 8, 2048, 8), (72, 200, 2056, 7), (16, 136, 2040, 32),
                                                     (64, 64, 64, 1), (200, 72, 4096, 5)])
def test_split_matches_the_product(dtype, layout, m, n, k, splits) -> None:
    """Against float64: one rounding to the dtype (2^-11 or 2^-8 of the value), plus float32 sums of
    K products (K 2^-24 of the sum of their magnitudes)."""
    generator = torch.Generator("cuda").manual_seed(5)
    a = torch.randn((m, k) if layout[0] == "n" else (k, m), device="cuda", generator=generator).to(dtype)
    b = torch.randn((k, n) if layout[1] == "n" else (n, k), device="cuda", generator=generator).to(dtype)
    a, b = a if layout[0] == "n" else a.t(), b if layout[1] == "n" else b.t()
    out = _split(a, b, splits)
    exact, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    unit = 2.0**-11 if dtype == torch.float16 else 2.0**-8
    assert torch.all((out.double() - exact).abs() <= unit * exact.abs() + k * 2.0**-24 * size)
    assert torch.equal(out, _split(a, b, splits))


@pytest.mark.gpu
@pytest.mark.parametrize("n_odd", [False, True])
def test_split_of_ragged_columns_and_strided_output(n_odd: bool) -> None:
    """N % 4 != 0 (B stored K-contiguous) and an output of row stride > N: nothing past N is written."""
    m, n, k = 33, 67 if n_odd else 68, 4096
    generator = torch.Generator("cuda").manual_seed(6)
    a = torch.randn(m, k, device="cuda", generator=generator).half()
    b = torch.randn(n, k, device="cuda", generator=generator).half().t()
    full = torch.full((m, n + 5), 7.0, device="cuda", dtype=torch.float16)
    matmul.enqueue_split(a, b, full[:, :n], 9)
    assert torch.all(full[:, n:] == 7.0)
    exact, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    assert torch.all((full[:, :n].double() - exact).abs() <= 2.0**-11 * exact.abs() + k * 2.0**-24 * size)


@pytest.mark.gpu
@pytest.mark.parametrize(("m", "n", "k"), [(16, 6144, 4096), (1, 72, 5120), (130, 264, 8192)])
def test_split_variants_match_their_compositions_bitwise(m: int, n: int, k: int) -> None:
    """SwiGLU = swiglu of two products and row scales of one = the plain product, through the public
    entry points, which split here."""
    assert matmul.split_k(m, n, k) > 1
    generator = torch.Generator("cuda").manual_seed(7)
    x = torch.randn(m, k, device="cuda", generator=generator).bfloat16()
    gate, up = (torch.randn(k, n, device="cuda", generator=generator).bfloat16() for _ in range(2))
    value, gated = matmul.matmul_fp32acc(x, up), matmul.matmul_fp32acc(x, gate)
    assert torch.equal(matmul_swiglu.matmul_swiglu(x, gate, up), swiglu.swiglu(value, gated))
    ones = torch.ones(m, device="cuda")
    assert torch.equal(_split(x, gate, matmul.split_k(m, n, k), row_scale=ones), gated)
    scaled = rms_norm_matmul.rms_norm_matmul(x, gate)
    rstd = torch.rsqrt(x.double().square().mean(1, keepdim=True))
    exact = rstd * (x.double() @ gate.double())
    assert (scaled.double() - exact).norm() <= 2.0**-8 * exact.norm()


@pytest.mark.gpu
def test_split_replays_in_a_graph() -> None:
    """The sums' workspace belongs to the graph: every replay gives the eager result."""
    x = torch.randn(16, 8192, device="cuda").bfloat16()
    w = torch.randn(8192, 1024, device="cuda").bfloat16()
    assert matmul.split_k(16, 1024, 8192) > 1
    eager = matmul.matmul_fp32acc(x, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = matmul.matmul_fp32acc(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(matmul.matmul_fp32acc(x, w), eager)


@pytest.mark.gpu
def test_split_of_layouts_without_dma_runs_unsplit() -> None:
    x, w = torch.randn(16, 8192, device="cuda").half()[:, ::2], torch.randn(4096, 257, device="cuda").half()
    out = _split(x, w, 8)
    assert (out.double() - x.double() @ w.double()).norm() <= 2.0**-11 * (x.double() @ w.double()).norm()


@pytest.mark.parametrize(("splits", "workspace", "scale", "message"), [
    (0, 1 << 20, None, "splits"), (3, 1 << 20, None, "splits"), (2, (1 << 20) + 4, None, "aligned"),
    (2, 1 << 20, 1 << 20, "either")])
def test_split_rejects_before_any_launch(splits, workspace, scale, message) -> None:
    p = 1 << 20
    with pytest.raises(_hip.HipLibraryError, match=message):
        _hip.call("tk_gemm_splitk", 1, p, p, p if scale else None, scale, p, workspace, 64, 64, 128, splits,
                  128, 1, 64, 1, 64, 1, 64, 1, None)
