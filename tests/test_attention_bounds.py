"""GPU checks that a head or a packed sequence reads nothing of its neighbours: with NaN and infinities
in every other head (sequence), whose rows follow its own in memory, its outputs and gradients keep
their bits. Key blocks past a ragged end reach the kernels as zeros by the buffer range check alone
(P = 0 there, but 0 * NaN is NaN)."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab import _hip
from tklab.kernels.flash_attention import grouped_query_attention, varlen_attention

pytestmark = pytest.mark.gpu


def _poisoned(tensors, hide):
    """Copies whose hidden parts are NaN, infinite or huge by turns."""
    out = []
    for t in tensors:
        c = t.clone()
        bad = torch.full_like(c[hide], float("nan"))
        bad.view(-1)[1::3] = float("inf")
        bad.view(-1)[2::3] = -3e4
        c[hide] = bad
        out.append(c)
    return out


def _step(attend, q, k, v, do):
    q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
    out = attend(q, k, v)
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), do))


# One head size and mask per kernel and workgroup (rows), N no multiple of 64 keys.
@pytest.mark.parametrize(("dim", "causal", "batch", "heads", "kv_heads", "n", "rows"), [
    (64, True, 1, 8, 4, 333, 64), (64, False, 1, 8, 4, 333, 64), (128, True, 1, 8, 4, 100, 64),
    (128, False, 1, 8, 4, 129, 64), (64, True, 20, 16, 4, 250, 128), (128, True, 10, 16, 4, 250, 128),
    (128, False, 1, 26, 26, 1050, 128), (64, True, 130, 16, 8, 250, 256), (64, False, 12, 16, 4, 250, 256),
    (128, True, 36, 16, 4, 250, 256), (128, False, 12, 16, 4, 250, 256),
])
def test_heads_do_not_see_the_next_head(dim, causal, batch, heads, kv_heads, n, rows) -> None:
    assert _hip.query("tk_attn_fwd_rows", batch, heads, kv_heads, n, dim, 0, int(causal)) == rows
    g = torch.Generator("cuda").manual_seed(n + dim)
    q, do = (torch.randn(batch, heads, n, dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(batch, kv_heads, n, dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    group = heads // kv_heads
    kv_odd = torch.arange(kv_heads, device="cuda") % 2 == 1
    odd = kv_odd.repeat_interleave(group)

    def attend(q, k, v):
        return grouped_query_attention(q, k, v, causal=causal)

    want = _step(attend, q, k, v, do)
    q2, do2 = _poisoned((q, do), (slice(None), odd))
    k2, v2 = _poisoned((k, v), (slice(None), kv_odd))
    got = _step(attend, q2, k2, v2, do2)
    for a, b, hidden in zip(got, want, (odd, odd, kv_odd, kv_odd)):
        assert torch.isfinite(b).all()
        assert bits_equal(a[:, ~hidden], b[:, ~hidden])


@pytest.mark.parametrize(("dim", "causal", "lengths", "rows"), [
    (64, True, [333, 70, 129, 1, 65, 40], 64), (128, True, [100, 333, 65, 64], 64),
    (64, False, [129, 65, 333, 1], 64), (128, False, [100, 33, 65, 64], 64),
    (64, True, [250, 129, 1, 257] * 12, 128), (128, True, [1000, 77, 500, 900], 128),
    (128, False, [300, 20, 130, 100] * 10, 128), (64, False, [1000, 1025, 90, 80] * 3, 256),
    (128, True, [2900, 2600] * 2, 256), (128, False, [2000, 1, 999, 1100], 256),
])
def test_sequences_do_not_see_the_next_sequence(dim, causal, lengths, rows) -> None:
    heads, kv_heads, total = 16, 4, sum(lengths)
    assert _hip.query("tk_attn_fwd_rows", len(lengths), heads, kv_heads, max(lengths), dim, total,
                      int(causal)) == rows
    g = torch.Generator("cuda").manual_seed(total)
    q, do = (torch.randn(total, heads, dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(total, kv_heads, dim, device="cuda", generator=g).bfloat16() for _ in range(2))
    ends = torch.tensor([0, *lengths]).cumsum(0)
    cu = ends.to("cuda", torch.int32)
    hidden = torch.zeros(total, dtype=torch.bool, device="cuda")
    for first, last in list(zip(ends, ends[1:]))[1::2]:
        hidden[first:last] = True

    def attend(q, k, v):
        return varlen_attention(q, k, v, cu, max(lengths), causal=causal)

    want = _step(attend, q, k, v, do)
    got = _step(attend, *_poisoned((q, k, v, do), (hidden,)))
    for a, b in zip(got, want):
        assert torch.isfinite(b).all()
        assert bits_equal(a[~hidden], b[~hidden])
