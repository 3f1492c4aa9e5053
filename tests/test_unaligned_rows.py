"""GPU checks of the row kernels at any element boundary: odd widths, odd strides and offset bases,
with NaN around every row, so that a value read past its row's end shows in the result. Where
an aligned problem of the same width exists the bits must match it."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab.harness.tolerances import assert_close
from tklab.kernels.fused_softmax import online_softmax, softmax

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
# Around one vector, one wave's vectors, the row shapes' limits and a 16384-column chunk.
WIDTHS = [1, 3, 7, 8, 9, 15, 17, 63, 65, 255, 257, 511, 513, 1000, 1023, 1025, 2047, 4095, 4097,
          8191, 16383, 16385, 32001, 65535]


def _odd_rows(rows: int, cols: int, dtype: torch.dtype, seed: int, offset: int = 1) -> torch.Tensor:
    """(rows, cols) at element offset `offset`, row stride odd and at least cols + 2, in NaN."""
    stride = cols + 2 + cols % 2 + 1
    storage = torch.full((rows * stride + offset + 8,), float("nan"), device="cuda", dtype=dtype)
    view = storage[offset:offset + rows * stride].view(rows, stride)[:, :cols]
    g = torch.Generator("cuda").manual_seed(seed)
    view.copy_(torch.randn(rows, cols, device="cuda", generator=g) * 2)
    return view


def _tail(out: torch.Tensor, cols: int) -> torch.Tensor:
    """Elements of a NaN-filled output's storage outside its rows."""
    rows, stride = out.shape[0], out.stride(0)
    whole = torch.as_strided(out, (rows, stride), (stride, 1))
    return whole[:, cols:]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", WIDTHS)
def test_softmax(dtype, cols) -> None:
    x = _odd_rows(5, cols, dtype, seed=cols)
    want = torch.softmax(x.double(), dim=-1)
    for run in (softmax, online_softmax):
        assert_close(run(x), want)
        assert_close(run(x.contiguous()), want)
    aligned = torch.empty_like(x, memory_format=torch.contiguous_format).copy_(x)
    assert bits_equal(online_softmax(x), online_softmax(aligned))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [9, 250, 4099, 32769])
@pytest.mark.parametrize("offset", [1, 3])  # 3: every output row starts where its input row does
def test_softmax_writes_its_rows_only_and_keeps_infinities(dtype, cols, offset) -> None:
    from tklab.kernels.fused_softmax import _launch, _launch_online

    x = _odd_rows(4, cols, dtype, seed=cols, offset=3)
    x[1, :] = -float("inf")
    x[2, cols - 1] = float("inf")
    x[3, : cols - 1] = -float("inf")
    want = torch.softmax(x.double(), dim=-1)
    for launch in (_launch, _launch_online):
        out = _odd_rows(4, cols, dtype, seed=0, offset=offset)
        launch((x,), out)
        assert torch.isnan(_tail(out[:3], cols)).all()
        torch.testing.assert_close(out.double(), want, rtol=2e-2, atol=1e-3, equal_nan=True)


@pytest.mark.parametrize("cols", [16384 * 2 + 3, 16384 * 5 + 8, 70001])
def test_online_softmax_of_short_last_chunks(cols, monkeypatch) -> None:
    x = _odd_rows(3, cols, torch.bfloat16, seed=cols)
    got = online_softmax(x)
    assert_close(got, torch.softmax(x.double(), dim=-1))
    monkeypatch.setenv("TKLAB_ONLINE_SOFTMAX_POLLS", "0")
    assert bits_equal(online_softmax(x), got)
