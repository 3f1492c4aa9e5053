"""GPU checks of the small-workgroup attention forward kernels: the same heads get the same bits in
a small problem (16 queries per wave), inside larger ones (32 per wave, and the 256-query
workgroups) and in a variable-length batch."""

from __future__ import annotations

import pytest
import torch

from _helpers import bits_equal
from tklab.kernels.flash_attention import _launch_gqa_forward, rope_attention, varlen_attention

pytestmark = pytest.mark.gpu

# 64-query tiles of calls that take 16 queries per wave, 32 (causal) and 256 per workgroup
# (small_query_tiles, csrc/attention_fwd.hip).
TILES = (512, 1100, 8200)


def _forward(q, k, v, causal):
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:3], device="cuda", dtype=torch.float32)
    _launch_gqa_forward(q, k, v, out, lse, causal=causal)
    return out, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("n", [1, 15, 16, 63, 64, 65, 127, 129, 250, 333, 1000, 1100])
def test_same_bits_at_every_size(dtype, causal, dim, n) -> None:
    heads, kv = 8, 4
    per_batch = heads * -(-n // 64)
    batch = -(-TILES[2] // per_batch)
    g = torch.Generator("cuda").manual_seed(n + dim)
    # Scores large enough that the lazily moved softmax reference moves often.
    q, k, v = ((torch.randn(batch, h, n, dim, device="cuda", generator=g) * s).to(dtype)
               for h, s in ((heads, 4.0), (kv, 1.0), (kv, 1.0)))
    want = _forward(q, k, v, causal)
    for count in {max(1, TILES[0] // per_batch), -(-TILES[1] // per_batch)}:
        got = _forward(q[:count], k[:count], v[:count], causal)
        for small, large in zip(got, want):
            assert bits_equal(small, large[:count])


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("longest", [300, 2048, 2500, 4500])
def test_variable_lengths(causal, dim, longest) -> None:
    lengths = [longest, 1, 0, 130, 64, 700 % longest, 33]
    heads, kv = 16, 4
    g = torch.Generator("cuda").manual_seed(longest)
    q, k, v = (torch.randn(sum(lengths), h, dim, device="cuda", generator=g).bfloat16()
               for h in (heads, kv, kv))
    ends = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    cu = torch.tensor(ends, device="cuda", dtype=torch.int32)
    got = varlen_attention(q, k, v, cu, longest, causal=causal)
    for first, last in zip(ends, ends[1:]):
        if first == last:
            continue
        one = [t[first:last].transpose(0, 1)[None].contiguous() for t in (q, k, v)]
        want = _forward(*one, causal)[0][0].transpose(0, 1)
        assert bits_equal(got[first:last], want)


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
