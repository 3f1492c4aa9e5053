"""GPU checks of the row kernels at any element boundary where a wave's or a group's vectors end: rows
of at most one vector per lane, rows whose last vectors leave whole waves empty, and rows a few columns
short of a row shape's width. The rows lie in NaN-filled storage."""

from __future__ import annotations

import pytest
import torch

from tklab.harness.tolerances import assert_close
from tklab.kernels.fused_softmax import softmax
from test_unaligned_rows import DTYPES, _norm_step, _odd_rows

pytestmark = pytest.mark.gpu


def _check_norm(dtype, rows, cols) -> None:
    x, r, ds, dy = (_odd_rows(rows, cols, dtype, seed=i) for i in range(1, 5))
    w = _odd_rows(2, cols, dtype, seed=9)[0]
    s, y, rstd, dx, dw = _norm_step(x, r, w, ds, dy)
    s64 = s.double()
    torch.testing.assert_close(rstd.double(), torch.rsqrt(s64.square().mean(-1) + 1e-6), rtol=1e-5, atol=0)
    unit, g = s64 * rstd.double()[:, None], dy.double() * w.double()
    assert_close(y, unit * w.double())
    assert_close(dx, rstd.double()[:, None] * (g - unit * (g * unit).mean(-1, keepdim=True)) + ds.double())
    want = (dy.double() * unit).sum(0)
    # One rounding of the result; its float32 sums add less (rows 2^-24).
    assert (dw.double() - want).norm() / want.norm() < (1e-5 if dtype == torch.float32 else 1e-2)


# 64 lanes of one vector: 256 float32 or 512 16-bit columns.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [11, 64, 127, 248, 255, 256, 257, 264, 504, 511, 512, 513, 520])
def test_norm_of_one_vector_per_lane(dtype, cols) -> None:
    _check_norm(dtype, 601, cols)


# Rows of 256 and 1024 threads: one column short of, at and past the columns of whole waves, whole
# vectors of the group and half of its values.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [1027, 1279, 1281, 1535, 1537, 2047, 2559, 3071, 4093, 4351, 4353, 4607,
                                  4609, 5121, 8183, 8705, 12289, 16379])
def test_norm_of_waves_past_the_row(dtype, cols) -> None:
    if cols * torch.empty((), dtype=dtype).element_size() <= 65536:
        _check_norm(dtype, 259, cols)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [3, 4097])  # pairs of rows per wave from 4096 on
@pytest.mark.parametrize("cols", [9, 16, 127, 248, 255, 256, 257, 504, 511, 512, 513])
def test_softmax_of_one_vector_per_lane(dtype, rows, cols) -> None:
    x = _odd_rows(rows, cols, dtype, seed=cols)
    x[0, :] = -float("inf")
    x[1, : cols - 1] = -float("inf")
    x[2, cols - 1] = float("inf")
    torch.testing.assert_close(softmax(x).double(), torch.softmax(x.double(), -1), rtol=2e-2, atol=1e-3,
                               equal_nan=True)
    assert_close(softmax(x)[3:], torch.softmax(x[3:].double(), -1))


# A few columns short of a row shape of 1024 threads, where the shifted row would need the next one,
# and where it just fits.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [16377, 16381, 16383, 16385, 32761, 32765, 32767, 65529, 65533])
def test_contiguous_softmax_at_the_end_of_a_row_shape(dtype, cols) -> None:
    storage = torch.full((5 * cols + 8,), float("nan"), device="cuda", dtype=dtype)
    x = storage[3:3 + 5 * cols].view(5, cols)
    x.copy_(torch.randn(5, cols, device="cuda", generator=torch.Generator("cuda").manual_seed(cols)) * 3)
    assert_close(softmax(x.contiguous().clone()), torch.softmax(x.double(), -1))
    assert_close(softmax(x), torch.softmax(x.double(), -1))
