"""The rule that picks the attention forward's workgroup (``tk_attn_fwd_rows``): the sizes it was
measured at, and the same bits from each choice it makes for a packed batch."""

from __future__ import annotations

import random

import pytest
import torch

from _helpers import bits_equal
from tklab import _hip
from tklab.kernels.flash_attention import _launch_gqa_forward, varlen_attention


def _rows(heads: int, kv_heads: int, lengths: list[int], dim: int, causal: bool, *, packed: bool) -> int:
    longest, total = max(lengths), sum(lengths) if packed else 0
    return _hip.query("tk_attn_fwd_rows", len(lengths), heads, kv_heads, longest, dim, total, int(causal))


# (query heads, KV heads, lengths, head_dim, causal): rows of the workgroup that was the fastest, or
# within 4 % of it (csrc/attention_fwd.hip, small_query_tiles).
PACKED = [
    # Longest of one length on a full chip: the 256-query kernel is 3 to 22 % faster.
    ((32, 8, [2048] * 16, 128, True), 256), ((32, 8, [4096] * 8, 128, True), 256),
    ((32, 8, [4096], 128, True), 256), ((8, 8, [1024] * 64, 128, True), 256),
    ((8, 8, [2048] * 32, 128, True), 256), ((32, 32, [1000] * 32, 128, True), 256),
    ((32, 32, [768] * 40, 128, True), 256), ((8, 8, [1024] * 64, 64, True), 256),
    ((16, 16, [700] * 40, 64, True), 256),
    # Without a causal mask: 2 to 42 %.
    ((32, 8, [1024] * 32, 128, False), 256), ((32, 8, [2000] * 4, 128, False), 256),
    ((8, 8, [2048] * 32, 128, False), 256), ((32, 32, [768] * 40, 128, False), 256),
    ((32, 32, [256] * 100, 128, False), 256),
    # Padding of short and ragged sequences outweighs that.
    ((32, 8, [16] * 2000, 128, True), 128), ((32, 8, [300] * 100, 128, True), 128),
    ((32, 8, [1000] * 32, 128, True), 128), ((32, 32, [300] * 100, 128, True), 128),
    ((32, 8, [64] * 500, 128, False), 128), ((16, 16, [256] * 100, 128, False), 128),
    ((32, 8, [640] * 50, 64, True), 128), ((32, 16, [386] * 27, 128, True), 128),
    ((32, 8, [45, 90, 150, 300, 450, 500, 600, 700, 800, 900, 1000, 1200, 1600, 1857, 1808], 128, True), 128),
    ((16, 16, [300, 400, 500, 600, 700, 800, 900, 1000, 1100, 1200, 1500, 1800, 350, 450, 900], 64, True), 128),
    # A last round of 256-query workgroups that leaves half of the compute units idle, and none.
    ((32, 32, [862, 500, 620], 128, False), 128), ((32, 32, [500] * 12, 128, False), 256),
    ((16, 16, [500] * 12, 128, False), 128), ((16, 16, [1000] * 6, 128, False), 128),
    ((8, 4, [532] * 19, 128, False), 128), ((8, 8, [500] * 12, 128, False), 256),
    ((8, 8, [1000] * 6, 128, False), 256), ((32, 8, [1000] * 4, 128, False), 256),
    # Few tiles leave compute units idle.
    ((8, 8, [1000] * 4, 128, True), 64), ((8, 8, [4096], 64, True), 64), ((8, 8, [4096], 128, False), 128),
]


@pytest.mark.parametrize(("problem", "rows"), PACKED)
def test_packed_batches_take_the_measured_workgroup(problem, rows) -> None:
    assert _rows(*problem, packed=True) == rows


@pytest.mark.parametrize(("problem", "rows"), [
    ((16, 16, [1024], 64, True), 64), ((16, 16, [4096], 64, True), 64), ((16, 16, [8192], 64, True), 128),
    ((128, 128, [8192], 64, True), 256), ((32, 32, [1024], 128, True), 64), ((8, 8, [8192], 128, True), 128),
    ((256, 256, [512], 128, True), 128), ((64, 64, [2048], 128, True), 256), ((32, 32, [1024], 64, False), 64),
    ((64, 64, [1024], 64, False), 256), ((16, 16, [1024], 128, False), 64), ((4, 4, [8192], 128, False), 128),
    ((8, 8, [1000] * 16, 128, True), 128), ((4, 4, [1000] * 31, 128, True), 256),
    ((4, 4, [1000] * 27, 128, True), 128), ((1, 1, [900] * 113, 128, True), 256),
    ((1, 1, [768] * 141, 128, True), 128), ((48, 48, [512], 128, False), 64), ((64, 64, [1024], 128, False), 256),
])
def test_equal_lengths_take_the_fastest_column_of_the_table(problem, rows) -> None:
    assert _rows(*problem, packed=False) == rows


def test_every_size_has_a_workgroup() -> None:
    rng = random.Random(1)
    for _ in range(2000):
        kv = rng.choice([1, 2, 3, 8, 32])
        lengths = [rng.randint(1, 5000)] * rng.randint(1, 60)
        problem = (kv * rng.choice([1, 2, 4, 7]), kv, lengths, rng.choice([64, 128]), rng.random() < 0.5)
        rows = _rows(*problem, packed=rng.random() < 0.5)
        assert rows in ((64, 128, 256) if problem[3] == 128 or problem[4] else (64, 256))
    assert _hip.query("tk_attn_fwd_rows", 1, 8, 3, 64, 64, 0, 1) == 0


# Every (rows, head_dim, causal) a packed batch can take.
@pytest.mark.gpu
@pytest.mark.parametrize(("problem", "rows"), [
    ((8, 2, [130, 1, 65, 64], 64, True), 64), ((8, 8, [513, 200], 64, False), 64),
    ((8, 2, [127, 300], 128, True), 64), ((8, 8, [129, 63], 128, False), 64),
    ((16, 4, [200, 129, 1, 257] * 20, 64, True), 128), ((16, 8, [1000, 77, 500, 900], 128, True), 128),
    ((8, 8, [4030], 128, False), 128), ((16, 16, [256, 1, 129, 128] * 10, 128, False), 128),
    ((16, 4, [300, 20, 130] * 12, 128, False), 128), ((16, 16, [1024] * 40, 64, True), 256),
    ((16, 4, [1000, 1025, 90] * 3, 64, False), 256), ((8, 8, [1400, 1350] * 10, 128, True), 256),
    ((16, 4, [2000, 1, 999], 128, False), 256),
])
def test_packed_bits_do_not_depend_on_the_workgroup(problem, rows) -> None:
    heads, kv, lengths, dim, causal = problem
    assert _rows(*problem, packed=True) == rows
    total = sum(lengths)
    g = torch.Generator("cuda").manual_seed(total)
    q, k, v = (torch.randn(total, h, dim, device="cuda", generator=g).bfloat16() for h in (heads, kv, kv))
    ends = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    cu = torch.tensor(ends, device="cuda", dtype=torch.int32)
    got = varlen_attention(q, k, v, cu, max(lengths), causal=causal)
    checked = set()
    for first, last in zip(ends, ends[1:]):
        if last - first in checked:
            continue
        checked.add(last - first)
        one = [t[first:last].transpose(0, 1)[None].contiguous() for t in (q, k, v)]
        want = torch.empty_like(one[0])
        _launch_gqa_forward(*one, want, torch.empty(want.shape[:3], device="cuda"), causal=causal)
        assert bits_equal(got[first:last], want[0].transpose(0, 1))
