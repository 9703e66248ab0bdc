"""The classic launch's integer arithmetic, emulated on the CPU: the division by an invariant and the
32-bit split ranges, against Python's integers and the rule they restate."""

from __future__ import annotations

import random

import pytest


def make_div(d: int) -> tuple[int, int, int]:
    if d <= 1:
        return d, 0, 0
    bits = (d - 1).bit_length()
    mul = ((1 << (31 + bits)) // d + 1) & 0xFFFFFFFF
    assert (1 << (31 + bits)) // d + 1 < 1 << 32  # it fits the kernel's 32 bits
    return d, mul, bits - 1


def div_by(n: int, v: tuple[int, int, int]) -> int:
    return n if v[0] == 1 else ((n * v[1]) >> 32) >> v[2]


def test_division_by_an_invariant():
    r = random.Random(1)
    ds = [1, 2, 3, 5, 7, 31, 32, 33, 641, 4095, 4096, (1 << 16) + 1, (1 << 30) - 1, (1 << 30) + 1, (1 << 31) - 1]
    ds += [r.randrange(1, 1 << r.randrange(1, 32)) for _ in range(500)]
    for d in ds:
        v = make_div(d)
        top = (1 << 31) - 1
        ns = [0, 1, d - 1, d, d + 1, top, top // d * d, top // d * d - 1] + [r.randrange(1 << 31) for _ in range(50)]
        assert all(div_by(n, v) == n // d for n in ns if 0 <= n <= top), d


def split_range(seq_len, max_seq_len, splits, split):
    """The kernel's steps, every intermediate checked to fit 32 bits."""
    chunk = -(-((max_seq_len + 31) // 32) // splits)
    by_splits, by_chunk = make_div(splits), make_div(max(1, chunk))
    tiles = (seq_len + 31) >> 5
    if chunk and seq_len <= max_seq_len:
        n = div_by(tiles + chunk - 1, by_chunk)
    else:
        chunk = max(div_by(tiles + splits - 1, by_splits), chunk, 1)
        n = (tiles + chunk - 1) // chunk
    assert split * chunk < 1 << 32 and tiles << 5 < 1 << 32
    lo = min(split * chunk, tiles)
    return min(lo << 5, seq_len), min(min(lo + chunk, tiles) << 5, seq_len), max(1, n)


@pytest.mark.parametrize("seed", range(4))
def test_split_ranges(seed):
    r = random.Random(seed)
    for _ in range(3000):
        splits = r.choice([1, 2, 3, 7, 16, 64, 4096])
        seq_len = r.choice([0, 1, 31, 32, 33, r.randrange(1 << r.randrange(1, 32)), (1 << 31) - 1])
        longest = r.choice([0, seq_len, r.randrange(1 << r.randrange(1, 32)), (1 << 31) - 1])
        split = r.randrange(splits)
        # the rule: a chunk of whole 32-token tiles, of the sequence itself or of the longest one
        own = -(-(-(-seq_len // 32)) // splits)
        chunk = 32 * max(1, own, -(-(-(-longest // 32)) // splits))
        lo = min(split * chunk, seq_len)
        want = lo, min(lo + chunk, seq_len), max(1, -(-seq_len // chunk))
        assert split_range(seq_len, longest, splits, split) == want
