"""The f16 arithmetic of the tiled experts (csrc/tile_half.h), restated in numpy: what the operands keep of a row and of its
group sums. Every statement is about exact values, so float64 decides it.
"""
import numpy as np
import pytest


def scale(largest):
    """th_scale: the power of two that brings a finite row's largest value under 2^14."""
    e = int(np.float32(largest).view(np.uint32)) >> 23 & 0xff
    return np.uint32(min(13 - (e - 127), 126) + 127 << 23).view(np.float32)


def test_scale_of_every_exponent():
    for e in range(255):
        for mantissa in (0, 1, 0x7fffff):
            v = np.uint32(e << 23 | mantissa).view(np.float32)
            f = scale(v)
            assert 2.0 ** -126 <= f < np.inf and 2.0 ** -126 <= np.float32(1) / f < np.inf
            assert np.log2(np.float64(f)) % 1 == 0 and np.float32(1) / f * f == 1
            assert float(v) * float(f) < 2.0 ** 14
            if e > 13:  # above 2^-113 the whole of f16's range is used
                assert float(v) * float(f) >= 2.0 ** 13


def pieces(S):
    """th_sum: hi, and the two pieces of 2^11 (S / 64 - hi), as the two products add them up."""
    v = np.float32(S) * np.float32(0.015625)
    h = v.astype(np.float16)
    r = (v - h.astype(np.float32)) * np.float32(2048)
    r1 = r.astype(np.float16)
    r2 = (r - r1.astype(np.float32)).astype(np.float16)
    return h, r1, r2


def test_sums_keep_float32():
    """A group's sum (32 values under 2^14, so under 2^19): from 2^-6 up the pieces add up to all 24 bits of it, below that to
    2^-30; and every product with a minimum, m or m 2^-11 for m to 63, is exact in float32."""
    rng = np.random.default_rng(3)
    S = (rng.uniform(1, 2, 200000) * 2.0 ** rng.integers(-6, 19, 200000) * rng.choice([-1, 1], 200000)).astype(np.float32)
    h, r1, r2 = (x.astype(np.float64) for x in pieces(S))
    assert np.isfinite(h).all() and np.isfinite(r1).all()
    got = 64 * (h + (r1 + r2) * 2.0 ** -11)
    assert np.array_equal(got, S.astype(np.float64))
    small = (rng.uniform(-1, 1, 20000) * 2.0 ** -6).astype(np.float32)
    h0, a0, b0 = (x.astype(np.float64) for x in pieces(small))
    assert np.max(np.abs(64 * (h0 + (a0 + b0) * 2.0 ** -11) - small)) <= 2.0 ** -30
    two = 64 * (h + (S.astype(np.float64) / 64 - h).astype(np.float16))
    assert not np.array_equal(two, S.astype(np.float64)), "two pieces alone do not"
    m = np.arange(64)
    half = (m * 2.0 ** -11).astype(np.float16)
    assert np.array_equal(half.astype(np.float64), m * 2.0 ** -11)
    for x in (h, r1, r2):
        p = x[:2000, None] * half.astype(np.float64)
        assert np.array_equal(p.astype(np.float32).astype(np.float64), p)


@pytest.mark.parametrize("octaves", [0, 8, 16, 20])
def test_split_keeps_more_than_bf16(octaves):
    """hi + lo of a value `octaves` below its row's largest: never further off than bf16's hi + lo, down to 2^-20 of it."""
    rng = np.random.default_rng(octaves)
    x = (rng.uniform(1, 2, 100000) * 2.0 ** (13 - octaves)).astype(np.float32)
    h = x.astype(np.float16)
    lo = (x - h.astype(np.float32)).astype(np.float16)
    worst = np.max(np.abs(h.astype(np.float64) + lo - x) / x)

    def bf16(v):
        u = v.astype(np.float32).view(np.uint32)
        return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)
    b = bf16(x)
    b2 = bf16(x - b)
    assert worst <= max(2.0 ** -22, 2.0 ** (-39 + octaves + 1))
    assert worst <= np.max(np.abs(b.astype(np.float64) + b2 - x) / x)
