"""GPU checks of the 64-query attention forward kernel: bitwise the 256-query kernel's results,
which the same heads get inside a batch large enough for it."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab.kernels.flash_attention import _launch_gqa_forward, rope_attention

pytestmark = pytest.mark.gpu

# Most 64-query tiles of a call that takes the 64-query kernel (small_applies,
# csrc/attention_fwd.hip).
SMALL_TILES = 2048


def _forward(q, k, v, causal):
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:3], device="cuda", dtype=torch.float32)
    _launch_gqa_forward(q, k, v, out, lse, causal=causal)
    return out, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("n", [1, 15, 16, 63, 64, 65, 127, 129, 250, 333, 1000])
def test_same_bits_as_the_large_kernel(dtype, causal, dim, n) -> None:
    batch, heads, kv = -(-(SMALL_TILES + 1) // (8 * -(-n // 64))), 8, 4
    g = torch.Generator("cuda").manual_seed(n + dim)
    # Scores large enough that the lazily moved softmax reference moves often.
    q, k, v = ((torch.randn(batch, h, n, dim, device="cuda", generator=g) * s).to(dtype)
               for h, s in ((heads, 4.0), (kv, 1.0), (kv, 1.0)))
    assert batch * heads * -(-n // 64) > SMALL_TILES
    want = _forward(q, k, v, causal)
    for b in {0, batch - 1}:
        got = _forward(q[b:b + 1], k[b:b + 1], v[b:b + 1], causal)
        for small, large in zip(got, want):
            assert bits_equal(small[0], large[b])


@pytest.mark.parametrize("dim", [64, 128])
def test_rope_in_the_prologue(dim) -> None:
    n, batch = 200, 65
    g = torch.Generator("cuda").manual_seed(dim)
    q, k, v = (torch.randn(batch, 8, n, dim, device="cuda", generator=g).bfloat16() for _ in range(3))
    angle = torch.rand(n, dim // 2, device="cuda", generator=g) * 6
    cos, sin = angle.cos().bfloat16(), angle.sin().bfloat16()
    want = rope_attention(q, k, v, cos, sin, causal=True)
    got = rope_attention(q[3:4].contiguous(), k[3:4].contiguous(), v[3:4].contiguous(), cos, sin,
                         causal=True)
    assert bits_equal(got[0], want[3])
