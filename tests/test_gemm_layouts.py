"""GPU checks of tk_gemm on transposed operands and K tails: the same bits as the row-major
problem on contiguous copies (zero-padded to a multiple of 32 in K), with every operand a view
inside NaN-filled storage, so that a value read past its edge shows in the result."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal, dev, host, name
from oracle import oracle
from tklab.harness.tolerances import assert_close, assert_relative_frobenius
from tklab.kernels.matmul import matmul_fp32acc

pytestmark = pytest.mark.gpu

LAYOUTS = ["nn", "nt", "tn", "tt"]


def _view(rows: int, cols: int, dtype: torch.dtype, transposed: bool) -> torch.Tensor:
    """A (rows, cols) view, stored by rows or by columns, with NaN all round it."""
    shape = (cols, rows) if transposed else (rows, cols)
    storage = torch.full((shape[0] + 2, shape[1] + 16 + -shape[1] % 8), float("nan"),
                         device="cuda", dtype=dtype)
    inner = storage[1:1 + shape[0], 8:8 + shape[1]]
    inner.copy_(torch.randn(shape, device="cuda") * max(rows, cols) ** -0.25)
    return inner.t() if transposed else inner


def _padded(t: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    out = torch.zeros(rows, cols, device="cuda", dtype=t.dtype)
    out[:t.shape[0], :t.shape[1]] = t
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize(
    ("m", "n", "k"),
    [(8, 8, 8), (64, 72, 8), (256, 256, 32), (264, 520, 96), (520, 264, 1056), (72, 1032, 40),
     (264, 136, 232), (512, 512, 4096), (1000, 760, 1000)],
)
def test_same_bits_as_the_row_major_problem(dtype, layout, m, n, k) -> None:
    torch.manual_seed(m + n + k)
    a = _view(m, k, dtype, layout[0] == "t")
    b = _view(k, n, dtype, layout[1] == "t")
    k32 = -(-k // 32) * 32
    want = matmul_fp32acc(_padded(a, m, k32), _padded(b, k32, n))
    got = matmul_fp32acc(a, b)
    assert bits_equal(got, want)
    assert_relative_frobenius(got, a.float() @ b.float(), max_relative_error=1e-2)


@pytest.mark.parametrize(("m", "n", "k"), [(264, 136, 1), (264, 136, 33), (512, 256, 1027),
                                           (8, 8, 31), (136, 520, 4000)])
def test_weight_gradient_of_an_odd_token_count(m, n, k) -> None:
    """x.t() @ dy: K is the token count, any number."""
    torch.manual_seed(k)
    x, dy = _view(k, m, torch.bfloat16, False), _view(k, n, torch.bfloat16, False)
    got = matmul_fp32acc(x.t(), dy)
    k32 = -(-k // 32) * 32
    assert bits_equal(got, matmul_fp32acc(_padded(x.t(), m, k32), _padded(dy, k32, n)))
    expected = dev(oracle.gemm(host(x.t()), host(dy), name(x.dtype)), got)
    assert_close(got, expected)


@pytest.mark.parametrize(("m", "n", "k"), [(1, 257, 64), (33, 65, 256), (257, 1000, 72), (513, 3, 512)])
def test_input_gradient_of_any_width(m, n, k) -> None:
    """dy @ w.t(): rows of both operands are K-contiguous, M and N any number."""
    torch.manual_seed(n)
    dy, w = _view(m, k, torch.float16, False), _view(n, k, torch.float16, False)
    got = matmul_fp32acc(dy, w.t())
    expected = dev(oracle.gemm(host(dy), host(w.t()), name(dy.dtype)), got)
    assert_close(got, expected)
    assert_relative_frobenius(got, expected, max_relative_error=1e-3)


def _odd_view(rows: int, cols: int, dtype: torch.dtype, layout: str) -> torch.Tensor:
    """A (rows, cols) view at an odd element offset and row stride, by rows ("n"), by columns
    ("t") or with a column stride of 3 ("s"), with NaN all round and between."""
    shape = (cols, rows) if layout == "t" else (rows, cols)
    step = 3 if layout == "s" else 1
    width = shape[1] * step + 3 + shape[1] * step % 2  # odd
    storage = torch.full((shape[0] + 2, width), float("nan"), device="cuda", dtype=dtype)
    inner = storage[1:1 + shape[0], 1:1 + shape[1] * step:step]
    inner.copy_(torch.randn(shape, device="cuda") * max(rows, cols) ** -0.25)
    return inner.t() if layout == "t" else inner


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", [*LAYOUTS, "sn", "ns", "ss", "st", "ts"])
@pytest.mark.parametrize(
    ("m", "n", "k"),
    [(1, 1, 1), (3, 5, 7), (65, 63, 64), (64, 129, 65), (129, 257, 193), (2047, 1500, 129),
     (700, 4099, 200), (4100, 4100, 66), (31, 1000, 1501)],
)
def test_unaligned_and_strided_operands(dtype, layout, m, n, k) -> None:
    """The register-staged kernel's three tiles: the bits of the aligned problem."""
    torch.manual_seed(m + n + k)
    a, b = _odd_view(m, k, dtype, layout[0]), _odd_view(k, n, dtype, layout[1])
    m8, n8, k32 = -(-m // 8) * 8, -(-n // 8) * 8, -(-k // 32) * 32
    want = matmul_fp32acc(_padded(a, m8, k32), _padded(b, k32, n8))[:m, :n]
    got = matmul_fp32acc(a, b)
    assert bits_equal(got, want)
    assert_close(got, a.float() @ b.float())
