"""The classic launch's integer arithmetic: the division by an invariant and the 32-bit split ranges,
against Python's integers and the rule they restate. First in Python, every intermediate checked to
fit 32 bits; then the header that the kernels include (csrc/launch_math.h), by the host compiler."""

from __future__ import annotations

import ctypes
import pathlib
import random
import subprocess

import pytest

from pagedattn._abi import PA_MAX_SPLITS


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

# --------------------------------------------------------------------------
# csrc/launch_math.h itself, which the kernels and their launch code include,
# built by the host compiler.
# --------------------------------------------------------------------------

SHIM = """
#include "launch_math.h"
extern "C" void divide(uint32_t d, const uint32_t *n, int count, uint32_t *out) {
  const Div v = make_div(d);
  for (int i = 0; i < count; ++i) out[i] = div_by(n[i], v);
}
extern "C" void ranges(int seq_len, int max_seq_len, int splits, const int *split, int count, int *out) {
  const SplitDiv s = split_div(max_seq_len, splits);
  for (int i = 0; i < count; ++i) {
    const SplitRange r = split_range(seq_len, s, split[i]);
    out[3 * i] = r.lo, out[3 * i + 1] = r.hi, out[3 * i + 2] = r.n;
  }
}
"""
TOP = (1 << 31) - 1


@pytest.fixture(scope="module")
def shipped(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch_math")
    (d / "shim.cpp").write_text(SHIM)
    csrc = pathlib.Path(__file__).resolve().parent.parent / "paged-decode-attention_amd" / "csrc"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{csrc}", str(d / "shim.cpp"),
                    "-o", str(d / "shim.so")], check=True)
    return ctypes.CDLL(str(d / "shim.so"))


def test_shipped_division(shipped):
    r = random.Random(2)
    ds = [1, 2, 3, 5, 7, 31, 32, 33, 641, 4095, 4096, (1 << 16) + 1, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, TOP]
    ds += [1 << i for i in range(31)] + [r.randrange(1, 1 << r.randrange(1, 32)) for _ in range(2000)]
    for d in ds:
        ns = [0, 1, d - 1, d, min(d + 1, TOP), TOP, TOP // d * d, max(0, TOP // d * d - 1)]
        ns += [r.randrange(1 << 31) for _ in range(50)]
        out = (ctypes.c_uint32 * len(ns))()
        shipped.divide(ctypes.c_uint32(d), (ctypes.c_uint32 * len(ns))(*ns), len(ns), out)
        assert list(out) == [n // d for n in ns], d


def test_shipped_split_ranges(shipped):
    """Whole chunks of 32-token tiles, of the sequence itself or of the longest one, at every edge of
    the 32-bit arithmetic; the ranges of a sequence's splits cover it once."""
    r = random.Random(3)
    edges = [0, 1, 31, 32, 33, TOP - 31, TOP - 1, TOP]
    for _ in range(6000):
        splits = r.choice([1, 2, 3, 7, 16, 64, 1000, 4096, PA_MAX_SPLITS])
        seq_len = r.choice([*edges, r.randrange(1 << r.randrange(1, 32))])
        longest = r.choice([0, seq_len, *edges, r.randrange(1 << r.randrange(1, 32))])
        which = sorted({0, 1 % splits, splits // 2, splits - 1, r.randrange(splits)})
        out = (ctypes.c_int * (3 * len(which)))()
        shipped.ranges(seq_len, longest, splits, (ctypes.c_int * len(which))(*which), len(which), out)
        own = -(-(-(-seq_len // 32)) // splits)
        chunk = 32 * max(1, own, -(-(-(-longest // 32)) // splits))
        n = max(1, -(-seq_len // chunk))
        assert n <= splits
        for i, split in enumerate(which):
            lo = min(split * chunk, seq_len)
            assert tuple(out[3 * i:3 * i + 3]) == (lo, min(lo + chunk, seq_len), n), (seq_len, longest, splits, split)
