"""Unsplit launches that start the longest sequences first: the order changes no result."""

from __future__ import annotations

import pytest
import torch

from helpers import max_abs, seeded_q
from oracle import reference as oracle
from pagedattn import ModelShape, allocate
from pagedattn.hip_decode import paged_decode_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_dtype", ["fp16", "fp8_e5m2", "int8"])
@pytest.mark.parametrize("hq,hkv,d,batch", [
    (8, 8, 32, 64),      # 512 workgroups: one round, not ordered
    (8, 8, 32, 65),      # the smallest ordered launch
    (14, 2, 64, 520),    # pairs of heads where the cache is 1-byte
    (40, 2, 64, 200),    # two head tiles
    (4, 1, 128, 1024),   # the largest order
    (4, 1, 128, 1025),   # one more: not ordered
])
def test_ordered_equals_unordered(kv_dtype, hq, hkv, d, batch):
    g = torch.Generator().manual_seed(81)
    lens = torch.randint(0, 90, (batch,), generator=g)
    lens[7] = 700
    c = allocate(ModelShape(hq, hkv, d, "o"), batch, lens.tolist(), kv_dtype=kv_dtype, seed=82, device="cuda")
    q = seeded_q(batch, hq, d, 83, device="cuda")
    a = torch.full_like(q, float("nan"))
    b = torch.full_like(q, float("nan"))
    paged_decode_hip(q, c, out=a, num_splits=1)
    paged_decode_hip(q, c, out=b, num_splits=1, seq_lens_host=lens.to(torch.int32))
    assert torch.equal(a, b)
    # lengths that are not the batch's give another order, and the same result
    paged_decode_hip(q, c, out=b, num_splits=1, seq_lens_host=torch.randint(0, 9999, (batch,), dtype=torch.int32))
    assert torch.equal(a, b)
    # ... and a tensor that cannot be an order is left alone, as before
    paged_decode_hip(q, c, out=b, num_splits=1, seq_lens_host=lens)
    assert torch.equal(a, b)


def test_default_call_of_a_ragged_batch():
    """The default call runs such a batch unsplit and ordered: it equals the unsplit launch."""
    g = torch.Generator().manual_seed(84)
    lens = torch.randint(32, 1023, (160,), generator=g).tolist()
    shape = ModelShape(64, 8, 128, "l")
    c = allocate(shape, 160, lens, seed=85, device="cuda", fill_device="cuda")
    q = seeded_q(160, 64, 128, 86, device="cuda")
    out = paged_decode_hip(q, c)
    assert torch.equal(out, paged_decode_hip(q, c, num_splits=1))
    rows = [0, 80, 159]
    from helpers import subset_cache

    want = oracle.reference_decode(q[rows].cpu(), subset_cache(c, rows), out_dtype=torch.float32)
    assert max_abs(out[rows], want) < 2e-3
