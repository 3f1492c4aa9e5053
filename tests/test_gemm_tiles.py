"""GPU checks of every tile of the DMA GEMM at ragged sizes: each layout against float32 math, the
same bits from every layout, and the fused variants bitwise their compositions."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab import _hip
from tklab.harness.tolerances import assert_close, assert_relative_frobenius
from tklab.kernels.matmul import launch_config, matmul_fp32acc
from tklab.kernels.matmul_swiglu import matmul_swiglu
from tklab.kernels.rms_norm_matmul import fold_norm_weight, rms_norm_matmul
from tklab.kernels.swiglu import swiglu

pytestmark = pytest.mark.gpu

# (tile, m, n, k): the smallest multiples of 8 found that pick each tile, all with ragged edges;
# K of one tile, of fewer tiles than a ring's stages and of many (half-used last tiles).
PROBLEMS = [
    ((64, 64), 8, 8, 32), ((64, 64), 72, 136, 1056), ((64, 64), 200, 1000, 4128),
    ((128, 64), 280, 3272, 96), ((64, 128), 416, 4224, 32), ((128, 128), 416, 4632, 160),
    ((128, 192), 824, 4632, 416), ((256, 128), 2184, 2728, 96), ((192, 128), 2456, 2320, 32),
    ((128, 256), 2320, 3272, 160), ((192, 192), 2320, 3408, 96), ((256, 256), 2320, 3680, 96),
]


def _operands(m, n, k, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    sc = k ** -0.25
    return [(torch.randn(s, device="cuda", generator=g) * sc).to(dtype)
            for s in ((m, k), (k, n), (k, n))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("tile", "m", "n", "k"), PROBLEMS)
def test_every_tile_in_every_layout(dtype, tile, m, n, k) -> None:
    a, b, _ = _operands(m, n, k, dtype, seed=m + n)
    config = launch_config(a, b)
    assert (config["block_m"], config["block_n"]) == tile
    c = matmul_fp32acc(a, b)
    want = a.float() @ b.float()
    assert_close(c, want)
    assert_relative_frobenius(c, want, max_relative_error=2e-3 if dtype == torch.bfloat16 else 1e-3)
    at, bt = a.t().contiguous().t(), b.t().contiguous().t()
    for left, right in ((a, bt), (at, b), (at, bt)):
        assert bits_equal(matmul_fp32acc(left, right), c)


@pytest.mark.parametrize(("tile", "m", "n", "k"), PROBLEMS)
def test_fused_variants_keep_the_bits_of_their_compositions(tile, m, n, k) -> None:
    x, gate, up = _operands(m, n, k, torch.bfloat16, seed=k)
    assert bits_equal(matmul_swiglu(x, gate, up), swiglu(matmul_fp32acc(x, up), matmul_fp32acc(x, gate)))
    out = torch.empty(m, n, device="cuda", dtype=x.dtype)
    ones = torch.ones(m, device="cuda")
    _hip.call("tk_gemm_rowscale", _hip.dtype_code(x.dtype), x.data_ptr(), gate.data_ptr(),
              ones.data_ptr(), out.data_ptr(), m, n, k, k, 1, n, 1, n, 1, _hip.stream_of(x))
    assert bits_equal(out, matmul_fp32acc(x, gate))
    weight = torch.ones(k, device="cuda", dtype=x.dtype)
    got = rms_norm_matmul(x, fold_norm_weight(weight, gate))
    rstd = torch.rsqrt(x.float().square().mean(-1, keepdim=True) + 1e-5)
    assert_close(got, (x.float() @ gate.float()) * rstd)
