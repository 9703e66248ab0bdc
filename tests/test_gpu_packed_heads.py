"""The classic kernel on pairs of 64-element kv heads of a 1-byte cache (one wave takes both heads
as a row of 128) against the oracle, and against the same heads taken one by one."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from helpers import max_abs, seeded_q
from oracle import reference as oracle
from pagedattn import ModelShape, allocate, decode_partials
from pagedattn.hip_decode import paged_decode_hip

pytestmark = pytest.mark.gpu

KV = [("fp8_e5m2", None), ("int8", torch.float16), ("int8", torch.float32)]


def _cache(hq, hkv, lens, kv_dtype, scale_dtype, page=16, seed=61):
    kw = {} if scale_dtype is None else {"scale_dtype": scale_dtype}
    return allocate(ModelShape(hq, hkv, 64, "p"), len(lens), lens, block_size=page, kv_dtype=kv_dtype, seed=seed,
                    device="cuda", **kw)


def _rows(c, sel):
    return dataclasses.replace(c, block_table=c.block_table[sel].contiguous(), seq_lens=c.seq_lens[sel].contiguous())


@pytest.mark.parametrize("kv_dtype,scale_dtype", KV)
@pytest.mark.parametrize("hq,hkv,splits,page", [
    (14, 2, 1, 16),   # 14 of 16 columns
    (14, 2, 3, 32),
    (16, 2, 2, 16),   # all 16 columns
    (4, 4, 1, 64),    # two columns a pair, two pairs
    (24, 4, 4, 16),
])
def test_pairs_match_the_oracle_and_single_heads(kv_dtype, scale_dtype, hq, hkv, splits, page):
    batch = -(-192 // (hkv // 2 * splits))  # the smallest batch that packs
    r = torch.Generator().manual_seed(62)
    lens = torch.randint(1, 420, (batch,), generator=r).tolist()
    lens[:5] = [1, 31, 32, 33, 0]
    c = _cache(hq, hkv, lens, kv_dtype, scale_dtype, page)
    q = seeded_q(batch, hq, 64, 63, device="cuda")
    q[:, ::3] *= 3  # peaked heads next to flat ones
    kw = {"num_splits": splits, "max_seq_len": max(lens)}
    got = paged_decode_hip(q, c, **kw)
    want = oracle.reference_decode(q, c, out_dtype=torch.float32)
    assert bool((got[4] == 0).all())  # the empty sequence, for which the oracle has no value
    want[4] = 0
    assert max_abs(got, want) < 2e-3
    # one sequence fewer: every head by itself
    one = paged_decode_hip(q[1:].contiguous(), _rows(c, slice(1, None)), **kw)
    assert max_abs(got[1:], one) < 2e-3
    assert torch.equal(paged_decode_hip(q, c, **kw), got)
    part, lse = decode_partials(q, c, splits, max_seq_len=max(lens))
    part1, lse1 = decode_partials(q[1:].contiguous(), _rows(c, slice(1, None)), splits, max_seq_len=max(lens))
    assert torch.equal(torch.isinf(lse[1:]), torch.isinf(lse1))
    held = ~torch.isinf(lse1)
    assert max_abs(lse[1:][held], lse1[held]) < 2e-3 and max_abs(part[1:], part1) < 2e-3


@pytest.mark.parametrize("kv_dtype,scale_dtype", KV)
def test_one_token_rows_are_the_dequantised_v_rows(kv_dtype, scale_dtype):
    c = _cache(14, 2, [1] * 200, kv_dtype, scale_dtype)
    out = paged_decode_hip(seeded_q(200, 14, 64, 64, device="cuda"), c, num_splits=1)
    from pagedattn import dequantize_kv

    first = c.block_table[:, 0].long()
    # (index the raw bytes: fp8 tensors do not take every index kernel)
    rows = c.v_cache.view(torch.uint8)[first, 0].view(c.v_cache.dtype)
    v = dequantize_kv(rows, None if c.v_scale is None else c.v_scale[first, 0], kv_dtype)
    assert torch.equal(out, v.repeat_interleave(7, dim=1))


@pytest.mark.parametrize("what", ["k", "v"])
def test_infinities_of_one_head_stay_in_it(what):
    """An infinity in head 0's K or V (fp8 overflow) changes nothing of head 1's output."""
    c = _cache(14, 2, [50] * 192, "fp8_e5m2", None)
    q = seeded_q(192, 14, 64, 65, device="cuda")
    clean = paged_decode_hip(q, c, num_splits=1)
    store = (c.k_cache if what == "k" else c.v_cache).view(torch.uint8)
    store[c.block_table[3, 1].long(), 2, 0, 5] = 0x7C  # +inf, head 0, sequence 3
    got = paged_decode_hip(q, c, num_splits=1)
    assert torch.equal(got[:, 7:], clean[:, 7:])
    assert torch.equal(got[:3], clean[:3]) and torch.equal(got[4:], clean[4:])
    assert not bool(torch.isfinite(got[3, :7]).all())


@pytest.mark.parametrize("form", ["odd heads", "group 9", "head stride", "scale stride", "scale offset"])
def test_forms_that_do_not_pair(form):
    """Geometries outside the pairing rule give the oracle's result as before."""
    lens = [5, 70, 33] * 70
    if form == "odd heads":
        c = _cache(6, 3, lens, "int8", torch.float16)
    elif form == "group 9":
        c = _cache(18, 2, lens, "int8", torch.float32)
    else:
        c = _cache(4, 2, lens, "int8", torch.float16)
        if form == "head stride":  # heads 128 bytes apart
            wide = [torch.zeros((*t.shape[:3], 128), dtype=t.dtype, device="cuda") for t in (c.k_cache, c.v_cache)]
            for w, t in zip(wide, (c.k_cache, c.v_cache)):
                w[..., :64] = t
            c = dataclasses.replace(c, k_cache=wide[0][..., :64], v_cache=wide[1][..., :64])
        else:  # three scales a token, or a first scale at an odd half word
            wide = [torch.zeros((*t.shape[:2], 3), dtype=t.dtype, device="cuda") for t in (c.k_scale, c.v_scale)]
            at = 0 if form == "scale stride" else 1
            for w, t in zip(wide, (c.k_scale, c.v_scale)):
                w[..., at:at + 2] = t
            c = dataclasses.replace(c, k_scale=wide[0][..., at:at + 2], v_scale=wide[1][..., at:at + 2])
    q = seeded_q(len(lens), c.shape.num_q_heads, 64, 66, device="cuda")
    got = paged_decode_hip(q, c, num_splits=1)
    assert max_abs(got, oracle.reference_decode(q, c, out_dtype=torch.float32)) < 2e-3


@pytest.mark.parametrize("form", ["contiguous", "head stride", "scale offset"])
@pytest.mark.parametrize("entry", ["default", "planned", "noalloc"])
def test_launch_of_a_cache_that_does_not_pair(monkeypatch, form, entry):
    """A batch planned for pairs runs on them where the cache's layout pairs and otherwise takes the
    launch without them: the flat split here."""
    from pagedattn import hip_decode, plan_launch
    from pagedattn.hip_decode import decode_noalloc

    lens = [1500 + (i * 37) % 500 for i in range(256)]
    c = _cache(14, 2, lens, "int8", torch.float16)
    if form == "head stride":  # heads 128 bytes apart
        wide = [torch.zeros((*t.shape[:3], 128), dtype=t.dtype, device="cuda") for t in (c.k_cache, c.v_cache)]
        for w, t in zip(wide, (c.k_cache, c.v_cache)):
            w[..., :64] = t
        c = dataclasses.replace(c, k_cache=wide[0][..., :64], v_cache=wide[1][..., :64])
    elif form == "scale offset":  # scales at odd half words
        wide = [torch.zeros((*t.shape[:2], 3), dtype=t.dtype, device="cuda") for t in (c.k_scale, c.v_scale)]
        for w, t in zip(wide, (c.k_scale, c.v_scale)):
            w[..., 1:] = t
        c = dataclasses.replace(c, k_scale=wide[0][..., 1:], v_scale=wide[1][..., 1:])
    wps = hip_decode.flat_waves_per_simd("int8", 64, torch.float16)
    plan = plan_launch(256, 0, 2, 7, hip_decode._cu_count(c.k_cache.device), wps, kv_dtype="int8", head_dim=64,
                       seq_lens=lens)
    assert plan.packed_splits and plan.flat_splits
    launched = []
    real = hip_decode._launch
    monkeypatch.setattr(hip_decode, "_launch", lambda t, fn, a: launched.append(
        (a.num_splits, a.flat_splits, a.flat_seq_cost)) or real(t, fn, a))
    q = seeded_q(256, 14, 64, 67, device="cuda")
    if entry == "default":
        got = paged_decode_hip(q, c)
    elif entry == "planned":
        got = paged_decode_hip(q, c, **plan.launch_kwargs())
    else:
        got = decode_noalloc(q, c, torch.empty_like(q), **plan.launch_kwargs())
    want = (plan.packed_splits, 0, 0) if form == "contiguous" else (1, plan.flat_splits, plan.flat_seq_cost)
    assert launched == [want]
    from helpers import subset_cache

    rows = [0, 100, 255]
    ref = oracle.reference_decode(q[rows].cpu(), subset_cache(c, rows), out_dtype=torch.float32)
    assert max_abs(got[rows], ref) < 2e-3


def _wide_table(c, tokens=512):
    """The same sequences under a block table for `tokens` tokens: room for lengths that pair."""
    bt = torch.zeros((c.block_table.shape[0], tokens // c.block_size), dtype=torch.int32, device="cuda")
    bt[:, :c.block_table.shape[1]] = c.block_table
    return dataclasses.replace(c, block_table=bt)


def _launch_pairs(monkeypatch):
    """Whether each launch from here on took pairs."""
    from pagedattn import hip_decode

    took, real = [], hip_decode._launch
    monkeypatch.setattr(hip_decode, "_launch", lambda t, fn, a: took.append(hip_decode._takes_pairs(a)) or real(t, fn, a))
    return took


@pytest.mark.parametrize("q_dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv_dtype,scale_dtype", KV)
@pytest.mark.parametrize("hq,hkv,splits,page", [
    (14, 2, 1, 16),
    (14, 2, 3, 32),
    (16, 2, 2, 16),
    (4, 4, 1, 64),
    (24, 4, 9, 16),   # folded by four waves a row
])
def test_pairs_of_long_chunks(monkeypatch, kv_dtype, scale_dtype, q_dtype, hq, hkv, splits, page):
    """At the smallest batch and chunk that pair, with sequences longer than max_seq_len among them
    (split by their own lengths), against the oracle and against single heads."""
    took = _launch_pairs(monkeypatch)
    batch, told = -(-192 // (hkv // 2 * splits)), 256 * splits + 1
    g = torch.Generator().manual_seed(68)
    lens = torch.randint(1, told + 1, (batch,), generator=g).tolist()
    lens[:6] = [1, 33, 0, told, told + 300, 2 * told]
    c = _cache(hq, hkv, lens, kv_dtype, scale_dtype, page)
    q = seeded_q(batch, hq, 64, 69, device="cuda").to(q_dtype)
    q[:, ::3] *= 3
    kw = {"num_splits": splits, "max_seq_len": told}
    got = paged_decode_hip(q, c, **kw)
    one = paged_decode_hip(q, c, **dict(kw, max_seq_len=told - 1))  # a token less: every head by itself
    assert took == [True, False]
    want = oracle.reference_decode(q, c, out_dtype=torch.float32)
    want[2] = 0
    # 2e-3 in fp16; a bf16 result is rounded to 8 bits, half an ulp of a value up to 8 is 2^-6
    tol = 2e-3 if q_dtype == torch.float16 else 2.0 ** -6 + 2e-3
    assert max_abs(got, want) < tol and max_abs(got, one) < 2 * tol
    assert torch.equal(paged_decode_hip(q, c, **kw), got)


@pytest.mark.parametrize("kv_dtype,scale_dtype", KV)
def test_paired_one_token_rows_are_the_dequantised_v_rows(monkeypatch, kv_dtype, scale_dtype):
    from pagedattn import dequantize_kv

    took = _launch_pairs(monkeypatch)
    c = _wide_table(_cache(14, 2, [1] * 200, kv_dtype, scale_dtype))
    out = paged_decode_hip(seeded_q(200, 14, 64, 64, device="cuda"), c, num_splits=1)
    first = c.block_table[:, 0].long()
    rows = c.v_cache.view(torch.uint8)[first, 0].view(c.v_cache.dtype)
    v = dequantize_kv(rows, None if c.v_scale is None else c.v_scale[first, 0], kv_dtype)
    assert took == [True] and torch.equal(out, v.repeat_interleave(7, dim=1))


@pytest.mark.parametrize("what", ["k", "v"])
def test_infinities_of_one_paired_head_stay_in_it(monkeypatch, what):
    took = _launch_pairs(monkeypatch)
    c = _wide_table(_cache(14, 2, [50] * 192, "fp8_e5m2", None))
    q = seeded_q(192, 14, 64, 65, device="cuda")
    clean = paged_decode_hip(q, c, num_splits=1)
    store = (c.k_cache if what == "k" else c.v_cache).view(torch.uint8)
    store[c.block_table[3, 1].long(), 2, 0, 5] = 0x7C  # +inf, head 0, sequence 3
    got = paged_decode_hip(q, c, num_splits=1)
    assert took == [True, True]
    assert torch.equal(got[:, 7:], clean[:, 7:])
    assert torch.equal(got[:3], clean[:3]) and torch.equal(got[4:], clean[4:])
    assert not bool(torch.isfinite(got[3, :7]).all())
