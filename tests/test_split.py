"""The three-part bf16 split of the prefill kernel's operands, on the CPU.

A statement of split_pair (flock_amd/csrc/prefill.hpp) in numpy: each part is what
is left, rounded to bf16. Checked for every significand of an f32, which decides
the sizes of the parts relative to the value.
"""
from __future__ import annotations

import numpy as np


def bf16(x: np.ndarray) -> np.ndarray:
    """f32 rounded to bf16, ties to even."""
    b = x.view(np.uint32)
    return ((b + np.uint32(0x7FFF) + ((b >> np.uint32(16)) & np.uint32(1)))
            & np.uint32(0xFFFF0000)).view(np.float32)


def split(x: np.ndarray) -> list[np.ndarray]:
    parts = []
    for _ in range(3):
        parts.append(bf16(x))
        x = x - parts[-1]
    assert not x.any()  # nothing is left: the parts add up to the value
    return parts


def test_parts_of_every_significand():
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32)
    p = [q.astype(np.float64) for q in split(x)]
    assert np.array_equal(p[0] + p[1] + p[2], x.astype(np.float64))
    assert np.max(np.abs(p[1]) / x) <= 2.0 ** -8
    assert np.max(np.abs(p[2]) / x) <= 2.0 ** -17
    # The three products that are left out, with the worst partner: 2 2^-8 2^-17 and a
    # bit, half an ulp of an f32 product; for a value times itself it is reached.
    left_out = np.abs(2 * p[1] * p[2] + p[2] * p[2]) / x.astype(np.float64) ** 2
    assert 2.0 ** -24.1 < left_out.max() < 2.0 ** -24 * (1 + 2.0 ** -8)


def test_values_from_2_to_minus_110_lose_nothing():
    # Parts end at 2^-133, bf16's smallest number.
    r = np.random.default_rng(1)
    x = ((1 + r.random(100000)) * r.choice((-1, 1), 100000) * 2.0 ** -110).astype(np.float32)
    p = split(x)
    ulp = 2.0 ** -133
    assert all(np.array_equal(np.round(q / ulp), q / ulp) for q in map(np.float64, p))
