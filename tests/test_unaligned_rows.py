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


def _norm_step(x, r, w, ds, dy):
    """Forward and backward through the private launchers into NaN-surrounded odd rows."""
    from tklab.kernels import residual_rms_norm as rrn
    from tklab.kernels import rms_norm as rn

    rows, cols = x.shape
    s, y = _odd_rows(rows, cols, x.dtype, 0), _odd_rows(rows, cols, x.dtype, 0, offset=5)
    rstd = torch.empty(rows, device="cuda")
    rrn._launch_forward(x, r, w, s, y, rstd, eps=1e-6, store_residual=True, store_stats=True)
    dx, dw = rn._launch_backward(dy, s, w, rstd, incoming_dx=ds)
    assert torch.isnan(_tail(s[:-1], cols)).all() and torch.isnan(_tail(y[:-1], cols)).all()
    return s, y, rstd, dx, dw


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("rows", "cols"), [(1, 3), (2, 8), (7, 9), (300, 65), (1000, 257), (513, 1023),
                                            (300, 1025), (260, 4097), (771, 2049), (3, 8193),
                                            (257, 16383), (2, 12345), (600, 1024)])
def test_residual_rms_norm(dtype, rows, cols) -> None:
    if cols * torch.empty((), dtype=dtype).element_size() > 65536:
        pytest.skip("row past the fused limit")
    x, r, ds, dy = (_odd_rows(rows, cols, dtype, seed=i) for i in range(1, 5))
    w = _odd_rows(2, cols, dtype, seed=9)[0]
    s, y, rstd, dx, dw = _norm_step(x, r, w, ds, dy)
    s64 = s.double()
    assert bits_equal(s, (x.float() + r.float()).to(dtype))
    rstd64 = torch.rsqrt(s64.square().mean(-1) + 1e-6)
    torch.testing.assert_close(rstd.double(), rstd64, rtol=1e-5, atol=0)
    unit, g = s64 * rstd64[:, None], dy.double() * w.double()
    assert_close(y, unit * w.double())
    assert_close(dx, rstd64[:, None] * (g - unit * (g * unit).mean(-1, keepdim=True)) + ds.double())
    want = (dy.double() * unit).sum(0)
    error = (dw.double() - want).norm() / want.norm()
    assert error < (1e-5 if dtype == torch.float32 else 1e-2), error
    if cols % 8 == 0:  # the same vectors as on aligned rows
        aligned = [t.contiguous().clone() for t in (x, r, w, ds, dy)]
        from tklab.kernels.residual_rms_norm import residual_rms_norm

        ax, ar, aw = (t.requires_grad_() for t in aligned[:3])
        as_, ay = residual_rms_norm(ax, ar, aw, 1e-6)
        adx, _, adw = torch.autograd.grad((as_, ay), (ax, ar, aw), aligned[3:])
        for got, same in ((s, as_), (y, ay), (dx, adx), (dw, adw)):
            assert bits_equal(got, same)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("rows", "cols"), [(1, 1), (1, 3), (1, 9), (3, 5), (7, 503), (8, 503), (179, 503),
                                            (1025, 1023), (5, 4096), (2, 16385)])
def test_swiglu_of_any_length(dtype, rows, cols) -> None:
    """Contiguous problems whose length ends inside a vector: the bits of the same elements in an
    aligned problem, nothing written past the end."""
    from tklab.kernels.swiglu import swiglu

    g = torch.Generator("cuda").manual_seed(rows * cols)
    count = rows * cols
    padded = -(-count // 64) * 64
    value, gate, dy = (torch.randn(padded, device="cuda", generator=g).to(dtype) for _ in range(3))

    def step(shape, *tensors):
        v, gt, d = (t.reshape(shape).detach().clone() for t in tensors)
        v.requires_grad_(), gt.requires_grad_()
        y = swiglu(v, gt)
        return (y, *torch.autograd.grad(y, (v, gt), d))

    whole = step((1, padded), value, gate, dy)
    for got, want in zip(step((rows, cols), value[:count], gate[:count], dy[:count]), whole):
        assert bits_equal(got.reshape(-1), want.reshape(-1)[:count])
