"""The planner's rules for pairs of kv heads, few-split classic launches and ordered batches, on both
sides of each line, and its plans against the library's own rules. CPU only."""

from __future__ import annotations

import ctypes
import random

import pytest

from pagedattn import _abi, plan_launch
from pagedattn.hip_decode import (
    CLASSIC_MARGIN_TILES,
    CLASSIC_MAX_CHUNK_TILES,
    CLASSIC_STREAM_LOSS,
    FEW_SPLIT_LONG_TILES,
    FEW_SPLIT_SHARE,
    FEW_SPLIT_SHARE_TILES,
    FEW_SPLITS_MAX,
    FEW_UNSPLIT_SHARE_TILES,
    MIN_SPLIT_TILES,
    ORDERED_MAX_BATCH,
    PACKED_MERGE_TILES,
    PACKED_SHARE,
    PACKED_SHARE_ONE_EACH,
    PACKED_SHORT_CHUNK_TILES,
    PACKED_SPLIT_MAX_RAGGED,
    PACKED_SPLIT_MIN_TILES,
    UNSPLIT_MARGIN_TILES,
    UNSPLIT_MAX_CHUNK_TILES,
    UNSPLIT_MAX_TILES,
    few_splits,
    ordered_batch_runs_unsplit,
    plan_num_splits,
)

FAKE = 0x10000  # 16-byte aligned, never dereferenced


def decode_args(batch, hq, hkv, kv, d=64, splits=1, **over):
    """pa_decode_args of a contiguous cache, as the library's checks see them."""
    a = _abi.PaDecodeArgs()
    a.q = a.k_cache = a.v_cache = a.out = a.block_table = a.seq_lens = a.part_out = a.part_lse = FAKE
    a.batch, a.num_q_heads, a.num_kv_heads, a.head_dim = batch, hq, hkv, d
    a.block_size, a.num_blocks, a.max_blocks, a.num_splits = 16, 64, 64, splits
    a.stride_qb, a.stride_qh = hq * d, d
    a.stride_kn, a.stride_kt, a.stride_kh = 16 * hkv * d, hkv * d, d
    a.stride_ob, a.stride_oh = hq * d, d
    a.stride_btb = 64
    a.kv_dtype = {"fp16": _abi.PA_KV_FP16, "bf16": _abi.PA_KV_BF16, "fp8_e5m2": _abi.PA_KV_FP8_E5M2,
                  "int8": _abi.PA_KV_INT8}[kv]
    a.scale_dtype = _abi.PA_SCALE_NONE
    if kv == "int8":
        a.k_scale = a.v_scale = FAKE
        a.scale_dtype, a.stride_sn, a.stride_st = _abi.PA_SCALE_FP16, 16 * hkv, hkv
    a.io_dtype = _abi.PA_IO_FP16
    a.sm_scale = d ** -0.5
    for k, v in over.items():
        setattr(a, k, v)
    return a


def pairs(a) -> bool:
    out = ctypes.c_int(-1)
    _abi.check(_abi.load().pa_decode_pairs(ctypes.byref(a), ctypes.byref(out)), "pa_decode_pairs")
    return bool(out.value)


@pytest.mark.parametrize("cus", [32, 64, 128, 256, 304])
def test_plans_for_pairs_get_pairs(cus):
    """Whatever the device's size, a plan cut for pairs of heads is one that the library runs on pairs."""
    r = random.Random(cus)
    packed = 0
    for _ in range(1500):
        batch, hi = r.randint(1, 600), int(2 ** r.uniform(6, 16))
        lens = [r.randint(max(1, hi // r.choice([1, 3])), hi) for _ in range(batch)]
        kv, hkv, group = r.choice([("fp8_e5m2", 2, 7), ("int8", 2, 7), ("int8", 4, 4), ("fp8_e5m2", 8, 8)])
        plan = plan_launch(batch, 0, hkv, group, cus, 2, kv_dtype=kv, head_dim=64, seq_lens=lens)
        if plan.packed_splits:
            packed += 1
            a = decode_args(batch, hkv * group, hkv, kv, splits=plan.packed_splits, max_seq_len=plan.max_seq_len,
                            max_blocks=-(-max(lens) // 16))
            assert pairs(a), (batch, hi, plan)
    assert packed > 100


def test_library_rule_for_pairs():
    ok = decode_args(192, 14, 2, "int8")
    assert pairs(ok)
    # one workgroup of pairs fewer than the library's least, counted over the splits
    assert not pairs(decode_args(191, 14, 2, "int8"))
    assert pairs(decode_args(64, 14, 2, "int8", splits=3)) and not pairs(decode_args(64, 14, 2, "int8", splits=2))
    # chunks of more than 256 tokens, of the longest sequence or of the block table's room for one
    assert pairs(decode_args(192, 14, 2, "int8", max_seq_len=257)) and not pairs(decode_args(192, 14, 2, "int8", max_seq_len=256))
    assert pairs(decode_args(64, 14, 2, "int8", splits=3, max_seq_len=769))
    assert not pairs(decode_args(64, 14, 2, "int8", splits=3, max_seq_len=768))
    assert pairs(decode_args(192, 14, 2, "int8", max_blocks=17)) and not pairs(decode_args(192, 14, 2, "int8", max_blocks=16))
    assert not pairs(decode_args(192, 14, 2, "int8", max_blocks=16, max_seq_len=9999))
    # types, head dims, head counts and groups
    assert pairs(decode_args(192, 14, 2, "fp8_e5m2")) and not pairs(decode_args(192, 14, 2, "fp16"))
    assert not pairs(decode_args(192, 14, 2, "int8", d=128)) and not pairs(decode_args(192, 14, 2, "int8", d=32))
    assert not pairs(decode_args(192, 6, 3, "int8")) and not pairs(decode_args(192, 18, 2, "int8"))
    assert pairs(decode_args(192, 16, 2, "int8"))
    # heads apart, a token stride under a pair, odd scales
    assert not pairs(decode_args(192, 14, 2, "int8", stride_kh=128, stride_kt=256, stride_kn=4096))
    assert not pairs(decode_args(192, 14, 2, "int8", stride_kt=64))
    assert not pairs(decode_args(192, 14, 2, "int8", k_scale=FAKE + 2))
    assert not pairs(decode_args(192, 14, 2, "int8", stride_st=3, stride_sn=48))
    # (the workspace has no say)
    assert pairs(decode_args(64, 14, 2, "int8", splits=3, part_out=None, part_lse=None))
    # a flat launch never does
    assert not pairs(decode_args(192, 14, 2, "int8", flat_splits=512))
    bad = ctypes.c_int(7)
    assert _abi.load().pa_decode_pairs(None, ctypes.byref(bad)) == _abi.PA_ERR_INVALID and bad.value == 0
    assert _abi.load().pa_decode_pairs(ctypes.byref(ok), None) == _abi.PA_ERR_INVALID


def test_plans_for_pairs_carry_the_launch_without_them():
    """A plan does not see the cache: the keywords of a launch cut for pairs hold the other one, too."""
    lens = [2048] * 256
    kw = dict(kv_dtype="int8", head_dim=64, seq_lens=lens)
    plan = plan_launch(256, 0, 2, 7, 256, 2, **kw)
    assert plan.packed_splits == 1 and plan.flat_splits > 0
    assert plan.launch_kwargs() == {"num_splits": 1, "max_seq_len": 2048,
                                    "unpaired": (plan.num_splits, plan.flat_splits, plan.flat_seq_cost)}
    # the same launch either way: nothing to carry
    short = plan_launch(512, 0, 2, 7, 256, 2, kv_dtype="int8", head_dim=64, seq_lens=[320] * 512)
    assert short.flat_splits == 0 and short.num_splits == 1 and "unpaired" not in short.launch_kwargs()


def test_the_bench_times_the_planned_launch():
    """Splits and flat ranges as the plan's keywords give them, cut for pairs of heads or not."""
    import pathlib
    import sys

    sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent))
    import bench

    plan = plan_launch(256, 0, 2, 7, 256, 2, kv_dtype="int8", head_dim=64, seq_lens=[2048] * 256)
    assert plan.packed_splits == 1 and plan.flat_splits > 0 and bench.planned_launch(plan) == (1, 0)
    plan = plan_launch(64, 0, 8, 4, 256, 2, kv_dtype="fp16", head_dim=128, seq_lens=[4096] * 64)
    assert bench.planned_launch(plan) == (1, plan.flat_splits) and plan.flat_splits > 0
    plan = plan_launch(1, 0, 8, 4, 256, 2, kv_dtype="fp16", head_dim=128, seq_lens=[2048])
    assert bench.planned_launch(plan) == (plan.num_splits, 0) and plan.num_splits > 1


def packed(lens, kv="int8", hkv=2, cus=256):
    return plan_launch(len(lens), 0, hkv, 7, cus, 2, kv_dtype=kv, head_dim=64, seq_lens=lens).packed_splits


@pytest.mark.parametrize("kv,batch,others,seen", [
    ("int8", 274, 100, {1, 0}), ("int8", 180, 120, {2, 0}), ("int8", 128, 200, {2, 0}), ("int8", 256, 200, {1, 0}),
    ("int8", 230, 100, {1, 2, 0}), ("fp8_e5m2", 274, 30, {1, 0}), ("fp8_e5m2", 190, 40, {2, 0}),
    ("fp8_e5m2", 64, 400, {4, 0}), ("fp8_e5m2", 256, 100, {1, 0}), ("fp8_e5m2", 200, 60, {1, 0})])
def test_pairs_instead_of_flat(kv, batch, others, seen):
    """Few workgroups: the fewest splits whose longest chunk is within its share, on both sides of the line."""
    def fits(splits, longest):
        share, more = (PACKED_SHARE_ONE_EACH if batch * splits <= 256 else PACKED_SHARE)[kv]
        most = share * (longest + (batch - 1) * others) / 256 + more - (PACKED_MERGE_TILES[kv] if splits > 1 else 0)
        uniform = longest <= 1.25 * (longest + (batch - 1) * others) / batch
        return -(-longest // splits) <= max(most, PACKED_SHORT_CHUNK_TILES if uniform else 0)

    got = set()
    for longest in range(others, 9 * others // 4):
        lens = [32 * longest] + [32 * others] * (batch - 1)
        choices = [s for s in (1, 2, 4) if batch * s >= 192 and (s == 1 or batch * s // 2 < 256)]
        want = next((s for s in choices if fits(s, longest)), 0)
        assert packed(lens, kv) == want, longest
        got.add(want)
    assert got >= seen


def test_pairs_limits():
    # many workgroups are taken up to PACKED_SPLIT_MAX_RAGGED times the mean, whatever the share
    n = 1000
    lens = [32 * 225] + [32 * 100] * (n - 1)
    for i in range(1, 126):
        lens[i] -= 32  # mean 100 tiles
    assert PACKED_SPLIT_MAX_RAGGED == 2.25 and max(lens) * n == 2.25 * sum(lens)
    assert packed(lens) == packed(lens, "fp8_e5m2") == 1
    lens[1] -= 1
    assert packed(lens) == packed(lens, "fp8_e5m2") == 0
    assert packed([32 * 220] + [32 * 100] * 512) == 1
    assert packed([32 * 220] + [32 * 100] * 511) == 0  # one fewer: the share's rule
    # more of them where a token's row is wide in fp8 (700 and 712 workgroups of 8 heads)
    assert packed([32 * 200] + [32 * 100] * 174, "fp8_e5m2", 8) == 0
    assert packed([32 * 200] + [32 * 100] * 177, "fp8_e5m2", 8) == 1
    assert packed([32 * 200] + [32 * 100] * 174, "int8", 8) == 1
    # 1-byte types only; the fewest splits, as a power of two, that give every CU a workgroup of pairs
    assert packed([8192] * 256, "fp16") == packed([8192] * 256, "bf16") == 0
    assert [packed([8192] * b) for b in (256, 250, 191, 128, 120, 95, 64, 60)] == [1, 1, 2, 2, 2, 4, 4, 4]
    # an unsplit launch with too few workgroups for pairs is cut in two from PACKED_SPLIT_MIN_TILES on
    t = 32 * PACKED_SPLIT_MIN_TILES
    assert packed([t] * 132) == 2 and packed([t - 32] * 132) == 0 and packed([t] * 127) == 0 and packed([t] * 192) == 0
    # where the flat split stands, pairs come before the few-workgroup classic split
    assert packed([5090] * 32) == 8 and classic([5090] * 32, "int8", 2, 7, 64) == 0


def classic(lens, kv, hkv, group, head_dim, known=True, cus=256):
    """Splits of the classic kernel in the batch's plan, 0 where it is flat."""
    p = plan_launch(len(lens), max(lens), hkv, group, cus, 2, kv_dtype=kv, head_dim=head_dim,
                    seq_lens=lens if known else None)
    return 0 if p.flat_splits else p.num_splits


def test_few_splits_keep_one_workgroup_a_cu():
    for batch, want in ((1, 32), (2, 16), (3, 10), (4, 8), (5, 6), (31, 1), (32, 1)):
        assert few_splits(batch, 16384, 8, 4, 256) == want
    # 16 heads a group are one tile, 17 are two
    assert few_splits(4, 16384, 8, 16, 256) == 8 and few_splits(4, 16384, 8, 17, 256) == 4
    # short sequences stay whole; from there chunks of MIN_SPLIT_TILES tiles at least
    whole = 32 * UNSPLIT_MAX_TILES
    assert few_splits(1, whole, 2, 7, 256) == 1
    assert few_splits(1, whole + 1, 2, 7, 256) == (UNSPLIT_MAX_TILES + 1) // MIN_SPLIT_TILES
    # FEW_SPLITS_MAX until each holds FEW_SPLIT_LONG_TILES tiles
    long = 32 * FEW_SPLITS_MAX * FEW_SPLIT_LONG_TILES
    assert few_splits(1, long, 2, 7, 256) == FEW_SPLITS_MAX
    assert few_splits(1, long + 32 * FEW_SPLIT_LONG_TILES, 2, 7, 256) == FEW_SPLITS_MAX + 1
    assert few_splits(1, 1 << 30, 1, 1, 1 << 20) == _abi.PA_MAX_SPLITS
    # more workgroups than CUs already
    assert few_splits(300, 16384, 8, 4, 256) == 1


@pytest.mark.parametrize("kv,hkv,group", [("fp16", 8, 4), ("bf16", 8, 4), ("fp8_e5m2", 8, 4), ("int8", 8, 8)])
def test_few_split_batches_without_lengths(kv, hkv, group):
    """Uniform or unknown lengths: classic while the longest chunk is within its limit."""
    for batch, splits, most in ((8, 4, CLASSIC_MAX_CHUNK_TILES[kv]), (32, 1, UNSPLIT_MAX_CHUNK_TILES[kv])):
        fits = 32 * splits * most
        for known in (False, True):
            assert classic([fits] * batch, kv, hkv, group, 128, known) == splits
            if splits > 1 or not known:  # (above it, known uniform lengths have rules of their own)
                assert classic([fits + 1] * batch, kv, hkv, group, 128, known) == 0
    # one workgroup more than CUs: the rule does not apply
    assert classic([32 * UNSPLIT_MAX_CHUNK_TILES[kv]] * 33, kv, hkv, group, 128, False) == 0


@pytest.mark.parametrize("kv,hkv,group", [("fp16", 8, 4), ("bf16", 8, 4), ("fp8_e5m2", 8, 4), ("int8", 8, 8)])
def test_few_split_ragged_batches(kv, hkv, group):
    """Known ragged lengths: classic while the longest chunk, CLASSIC_STREAM_LOSS slower, is within the
    margin over the tiles that the flat split gives a CU."""
    seen = set()
    rest = (140, 33) if kv == "int8" else (80, 20)  # tiles of the others: enough work for the flat split
    for batch, splits, margin, tiles in ((8, 4, CLASSIC_MARGIN_TILES[kv], rest[0]),
                                         (32, 1, UNSPLIT_MARGIN_TILES[kv], rest[1])):
        for longest in range(tiles, 3 * tiles):
            lens = [32 * longest] + [32 * tiles] * (batch - 1)
            if max(lens) <= 1.25 * sum(lens) / batch:
                continue  # nearly uniform
            a_cu = (longest + (batch - 1) * tiles) * 8 / 256
            want = splits if (1 + CLASSIC_STREAM_LOSS) * -(-longest // splits) <= a_cu + margin else 0
            assert classic(lens, kv, hkv, group, 128) == want, longest
            seen.add((splits, want))
    assert seen == {(4, 4), (4, 0), (1, 1), (1, 0)}


@pytest.mark.parametrize("batch,others", [(20, 5), (10, 8)])  # 160 and 80 workgroups unsplit
def test_batches_with_little_work(batch, others):
    """Too little for the flat split: few_splits, or the splits of plan_num_splits where the longest chunk
    is known to be far over a CU's share; without lengths few_splits."""
    seen = set()
    for longest in range(2 * others, 300):
        lens = [32 * longest] + [32 * others] * (batch - 1)
        few = few_splits(batch, max(lens), 8, 4, 256)
        more = FEW_UNSPLIT_SHARE_TILES if few == 1 else FEW_SPLIT_SHARE_TILES
        fits = -(-longest // few) <= FEW_SPLIT_SHARE * (longest + (batch - 1) * others) * 8 / 256 + more
        want = few if fits else plan_num_splits(lens, 8, 4, 256)[0]
        assert classic(lens, "fp16", 8, 4, 128) == want, longest
        seen.add((fits, want != few))
    assert seen >= {(True, False), (False, True)}
    assert classic([32 * 25] * 20, "fp16", 8, 4, 128, False) == few_splits(20, 800, 8, 4, 256) == 1


def ordered_lens(tiles, longest, others):
    """A batch of `tiles` tiles in all: one sequence of `longest`, the others of about `others`."""
    lens = [32 * longest] + [32 * others] * ((tiles - longest) // others)
    lens[-1] += 32 * (tiles - sum(n // 32 for n in lens))
    return lens


@pytest.mark.parametrize("kv,head_dim,hkv,group,rounds,longest,others", [
    ("fp16", 128, 8, 8, 2.5, 30, 14), ("bf16", 128, 8, 4, 2.5, 40, 12), ("fp16", 64, 8, 7, 1.0, 100, 20),
    ("fp16", 64, 8, 7, 2.0, 200, 60)])
def test_ordered_batches_by_rounds(kv, head_dim, hkv, group, rounds, longest, others):
    """Unsplit with the longest first: from `rounds` times the longest sequence's tiles of work a CU."""
    def ordered(lens, kv=kv, cus=256, hkv=hkv, group=group, head_dim=head_dim):
        return ordered_batch_runs_unsplit(lens, hkv, group, cus, kv, head_dim)

    lens = ordered_lens(int(rounds * longest * 256) // hkv, longest, others)
    assert len(lens) * hkv > 512 and ordered(lens)
    lens[-1] -= 32
    assert not ordered(lens)
    lens[-1] += 32
    # 1-byte types, unknown heads or lengths, a uniform batch
    assert not ordered(lens, kv="int8") and not ordered(lens, kv="fp8_e5m2") and not ordered(lens, kv=None)
    assert not ordered(lens, head_dim=None) and not ordered(None)
    assert not ordered([32 * longest] * len(lens))


def test_ordered_batches_by_size():
    def ordered(lens, hkv=8, group=8, cus=256, head_dim=128):
        return ordered_batch_runs_unsplit(lens, hkv, group, cus, "fp16", head_dim)

    # K/V a CU between the limits of the number of q heads (8 kv heads of 256 bytes, K and V: 16 bytes a
    # token and CU)
    def batch(tokens, longest, others):
        lens = [longest] + [others] * ((tokens - longest) // others)
        lens[1] += tokens - sum(lens)
        return lens

    for group, least, most in ((8, 256, 6144), (16, 256, 6144), (7, 512, 2048), (4, 512, 2048)):
        small, large = batch(least << 6, 90, 40), batch(most << 6, 900, 400)
        assert ordered(small, group=group) and ordered(large, group=group)
        small[2] -= 1
        large[2] += 1
        assert not ordered(small, group=group) and not ordered(large, group=group)
    lens = [600] + [200] * 400
    assert ordered(lens, group=4) and not ordered(lens, group=3) and not ordered(lens, group=1)
    # two workgroups a CU or fewer, and no fewer than the library orders on a smaller device
    few = [300] + [130] * 99
    assert not ordered(few[:64], cus=64) and ordered(few[:65], cus=64)
    # rows of 128 bytes: up to 1.5 MB a CU from one round on (above: two)
    rows = ordered_lens(100 * 256 // 8, 100, 20)
    assert ordered(rows, group=7, head_dim=64)
    # batches beyond the order's size
    many = [64] + [33] * (ORDERED_MAX_BATCH - 1)
    assert ordered(many) and not ordered(many + [33])
