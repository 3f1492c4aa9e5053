"""Order of the GEMM's sums and its workspace where K is split (``matmul.split_k``): which calls split,
whose bits follow from that, and that nothing is allocated for the calls that do not."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab.kernels import matmul
from tklab.kernels.matmul import matmul_fp32acc
from tklab.kernels.matmul_swiglu import matmul_swiglu
from tklab.kernels.swiglu import swiglu

SIZES = [(16, 1024, 8192), (33, 200, 5120), (64, 4096, 5120)]  # all split


@pytest.mark.parametrize(("shape", "strides", "taken"), [
    ((16, 64), (64, 1), True), ((16, 64), (72, 1), True), ((64, 16), (1, 64), True),
    ((16, 64), (65, 1), False), ((16, 63), (64, 1), False), ((16, 64), (128, 2), False),
    ((8, 1), (8, 1), False), ((8, 1), (1, 8), True), ((1 << 18, 4096), (4096, 1), False),
    ((1 << 18, 4088), (4096, 1), True),
])
def test_layouts_the_dma_kernels_take(shape, strides, taken) -> None:
    assert matmul._dma_operand(*shape, *strides) == taken


def _operands(m, n, k, seed=3):
    g = torch.Generator("cuda").manual_seed(seed)
    return [torch.randn(s, device="cuda", generator=g).bfloat16() for s in ((m, k), (k, n))]


def _odd(t: torch.Tensor) -> torch.Tensor:
    """The same values in rows that start at any element."""
    return torch.empty(t.shape[0], t.shape[1] + 1, device=t.device, dtype=t.dtype)[:, 1:].copy_(t)


def _whole(a, b):
    out = torch.empty(a.shape[0], b.shape[1], device=a.device, dtype=a.dtype)
    matmul._launch_fp32acc((a, b), out)
    return out


def _allocations(call) -> int:
    call()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    call()
    return torch.cuda.memory_stats()["allocation.all.allocated"] - before


@pytest.mark.gpu
@pytest.mark.parametrize(("m", "n", "k"), SIZES)
def test_bits_of_layouts_the_dma_does_not_take_are_the_unsplit_products(m, n, k) -> None:
    assert matmul.split_k(m, n, k) > 1
    a, b = _operands(m, n, k)
    want = _whole(a, b)
    for left, right in ((_odd(a), b), (a, _odd(b)), (_odd(a), _odd(b))):
        assert bits_equal(matmul_fp32acc(left, right), want)
        assert matmul.launch_config(left, right)["hip_kernel"] == "gemm_kernel"
    assert matmul.launch_config(a, b)["hip_kernel"] == "gemm_split_kernel"


@pytest.mark.gpu
@pytest.mark.parametrize(("m", "n", "k"), SIZES)
def test_a_row_has_the_same_bits_in_any_batch_of_an_unsplit_product(m, n, k) -> None:
    a, b = _operands(4096, n, k)
    assert matmul.split_k(4096, n, k) == 1
    assert bits_equal(_whole(a[:m], b), matmul_fp32acc(a, b)[:m])


@pytest.mark.gpu
def test_only_split_products_allocate_sums() -> None:
    m, n, k = SIZES[0]
    a, b = _operands(m, n, k)
    out = torch.empty(m, n, device="cuda", dtype=a.dtype)
    odd = _odd(a)
    assert _allocations(lambda: matmul._launch_fp32acc((a, b), out)) == 0
    assert _allocations(lambda: matmul._launch_fp16acc((a, b), out)) == 0
    assert _allocations(lambda: matmul_fp32acc(odd, b)) == 1  # the output
    assert _allocations(lambda: matmul_fp32acc(a, b)) == 2


@pytest.mark.gpu
def test_swiglu_composition_splits_as_its_products() -> None:
    """Transposed weights run unfused: two split products and SwiGLU."""
    m, n, k = SIZES[0]
    x, gate = _operands(m, n, k)
    up = _operands(m, n, k, seed=4)[1]
    gate_t, up_t = (w.t().contiguous().t() for w in (gate, up))
    want = matmul_swiglu(x, gate, up)
    assert bits_equal(matmul_swiglu(x, gate_t, up_t), want)
    assert bits_equal(swiglu(matmul_fp32acc(x, up), matmul_fp32acc(x, gate)), want)
