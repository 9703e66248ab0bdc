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


@pytest.mark.parametrize("host", ["equal", "two", "extreme", "negative", "steps"])
def test_any_host_lengths_make_an_order(host):
    """Whatever the lengths say, every sequence is taken once."""
    b = 700
    g = torch.Generator().manual_seed(87)
    c = allocate(ModelShape(4, 1, 32, "x"), b, torch.randint(0, 60, (b,), generator=g).tolist(), seed=88, device="cuda")
    q = seeded_q(b, 4, 32, 89, device="cuda")
    lens = {"equal": torch.full((b,), 9), "two": torch.arange(b) % 2 * 33,
            "extreme": torch.where(torch.arange(b) % 3 == 0, 2 ** 31 - 1, torch.arange(b) * 77 - 2 ** 31),
            "negative": -1 - 40 * torch.arange(b), "steps": torch.arange(b) * 255}[host].to(torch.int32)
    a, out = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    paged_decode_hip(q, c, out=a, num_splits=1)
    paged_decode_hip(q, c, out=out, num_splits=1, seq_lens_host=lens)
    assert torch.equal(a, out)


def test_captured_ordered_launch():
    """A captured launch keeps the order of the capture's host lengths: replays on other lengths, with
    eager work between them, equal eager launches."""
    b = 300
    g = torch.Generator().manual_seed(90)
    room = [400] * b
    c = allocate(ModelShape(8, 2, 64, "c"), b, room, seed=91, device="cuda", fill_device="cuda")
    q = seeded_q(b, 8, 64, 92, device="cuda")
    lens = torch.randint(1, 400, (b,), generator=g, dtype=torch.int32)
    c.seq_lens.copy_(lens)
    out = torch.empty_like(q)
    paged_decode_hip(q, c, out=out, num_splits=1, seq_lens_host=lens)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        paged_decode_hip(q, c, out=out, num_splits=1, seq_lens_host=lens)
    for _ in range(4):
        new = torch.randint(0, 400, (b,), generator=g, dtype=torch.int32)
        c.seq_lens.copy_(new)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        want = paged_decode_hip(q, c, num_splits=1)
        assert torch.equal(out, want)
        assert torch.equal(want, paged_decode_hip(q, c, num_splits=1, seq_lens_host=new))


@pytest.mark.parametrize("kv_dtype", ["fp16", "bf16", "fp8_e5m2", "int8"])
@pytest.mark.parametrize("hq,hkv,d,batch", [(8, 8, 32, 65), (14, 2, 64, 520), (40, 2, 64, 200), (4, 1, 128, 1024),
                                            (2, 1, 256, 600)])
def test_ordered_launches_of_long_sequences(kv_dtype, hq, hkv, d, batch):
    """Every geometry with a sequence long enough for an order, whatever its type."""
    g = torch.Generator().manual_seed(93)
    lens = torch.randint(0, 60, (batch,), generator=g)
    lens[batch // 3] = 1700
    c = allocate(ModelShape(hq, hkv, d, "o"), batch, lens.tolist(), kv_dtype=kv_dtype, seed=94, device="cuda")
    q = seeded_q(batch, hq, d, 95, device="cuda")
    a, b = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    paged_decode_hip(q, c, out=a, num_splits=1, max_seq_len=1700)
    paged_decode_hip(q, c, out=b, num_splits=1, max_seq_len=1700, seq_lens_host=lens.to(torch.int32))
    assert torch.equal(a, b)
