"""The merge by four waves a row (more than 8 splits; a flat split with 8 ranges a sequence or more)
at the edges of its passes and of its rule."""

from __future__ import annotations

import pytest
import torch

from helpers import max_abs, seeded_q
from oracle import reference as oracle
from pagedattn import LLAMA3_8B, allocate, split_reduce
from pagedattn.hip_decode import paged_decode_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("splits", [8, 9, 31, 32, 33, 64, 65, 300])
def test_split_reduce_edges(splits, d):
    """8 a wave, 32 a pass; rows with some splits empty, one left, and none left (zeros)."""
    g = torch.Generator().manual_seed(71)
    part = torch.randn((2, 3, splits, d), generator=g)
    lse = 20 * torch.randn((2, 3, splits), generator=g)
    lse[0, 1, ::3] = float("-inf")
    lse[1, 0, :] = float("-inf")
    lse[1, 0, splits - 1] = -3.0
    lse[1, 2, :] = float("-inf")
    part[torch.isinf(lse)] = 0
    got = split_reduce(part.cuda(), lse.cuda())
    want = oracle.split_merge(part, lse)
    want[1, 2] = 0
    # fp32 sums of at most 300 terms, then fp16: half an ulp of a value up to 8 is 2^-9
    assert max_abs(got, want) < 2.0 ** -9 + 1e-5


@pytest.mark.parametrize("batch,flat", [(8, 63), (8, 64), (8, 65), (3, 40), (1, 200)])
@pytest.mark.parametrize("kv_dtype", ["fp16", "int8"])
def test_flat_rule_edges(batch, flat, kv_dtype):
    """Either side of eight ranges a sequence, host tables and the GPU scan alike, empty rows zero."""
    lens = [(977 * i) % 3000 + 40 for i in range(batch)]
    if batch > 2:
        lens[1] = 0
    c = allocate(LLAMA3_8B, batch, lens, kv_dtype=kv_dtype, seed=72, device="cuda")
    q = seeded_q(batch, 32, 128, 73, device="cuda")
    a = paged_decode_hip(q, c, flat_splits=flat, seq_lens_host=torch.tensor(lens, dtype=torch.int32))
    b = paged_decode_hip(q, c, flat_splits=flat)
    assert torch.equal(a, b)
    want = oracle.reference_decode(q, c, out_dtype=torch.float32)
    if batch > 2:
        want[1] = 0
    assert max_abs(a, want) < 2e-3


@pytest.mark.parametrize("splits", [9, 33, 70])
def test_infinity_in_the_last_partial(splits):
    """The places of a pass past the last partial repeat its loads and count for nothing: an infinity
    there (an fp8 cache's overflow) stays one."""
    g = torch.Generator().manual_seed(74)
    part = torch.randn((1, 2, splits, 128), generator=g)
    part[0, 1, splits - 1, 5] = float("inf")
    lse = torch.randn((1, 2, splits), generator=g)
    got = split_reduce(part.cuda(), lse.cuda()).cpu()
    assert got[0, 1, 5] == float("inf") and int(torch.isfinite(got).sum()) == got.numel() - 1


@pytest.mark.parametrize("batch,heads", [(8, 32), (257, 1), (1 << 19, 32)])
def test_split_reduce_rows(batch, heads):
    """The most rows that four waves take, one more, and more rows than a launch of four waves each
    could hold (2^32 threads): all of them the same row here, its partials by stride 0."""
    g = torch.Generator().manual_seed(75)
    part, lse = torch.randn((1, 1, 9, 32), generator=g).cuda(), torch.randn((1, 1, 9), generator=g).cuda()
    got = split_reduce(part.expand(batch, heads, 9, 32), lse.expand(batch, heads, 9))
    want = oracle.split_merge(part.cpu(), lse.cpu())
    # fp32 sums of 9 terms, then fp16: half an ulp of a value up to 4 is 2^-10
    assert max_abs(got[:1, :1], want) < 2.0 ** -10 + 1e-5
    assert bool((got == got[0, 0]).all())


@pytest.mark.parametrize("d", [32, 128])
@pytest.mark.parametrize("splits", [9, 33])
def test_rows_of_empty_partials_are_zeros(splits, d):
    """Whatever the unused partials hold (uninitialised memory: NaN here)."""
    part, lse = torch.full((2, 3, splits, d), float("nan")), torch.full((2, 3, splits), float("-inf"))
    part[1, 2], lse[1, 2] = 1.5, 0.0
    got = split_reduce(part.cuda(), lse.cuda())
    assert bool((got[1, 2] == 1.5).all())
    got[1, 2] = 0
    assert bool((got == 0).all())
