"""The planner's native pass over host lengths against its numpy form, and every plan made from the
one against the plan made from the other."""

from __future__ import annotations

import ctypes
import random

import pytest
import torch

from pagedattn import _abi, flat_needs_merge, plan_launch
from pagedattn.hip_decode import _Lens


def _batches(seed):
    r = random.Random(seed)
    for _ in range(150):
        n = r.choice([0, 1, 2, 7, 64, 65, 300])
        hi = r.choice([1, 31, 32, 33, 1000, 70000])
        kind = r.choice(["same", "spread", "holes", "negative"])
        lens = [hi] * n if kind == "same" else [r.randint(0 if kind == "holes" else 1, hi) for _ in range(n)]
        if kind == "negative" and n:
            lens[r.randrange(n)] = -r.randint(1, 1 << 31)
        yield lens


@pytest.mark.parametrize("seed", range(3))
def test_native_stats_and_merge_equal_numpy(seed):
    r = random.Random(100 + seed)
    for lens in _batches(seed):
        a, b = _Lens(torch.tensor(lens, dtype=torch.int32)), _Lens(lens)
        assert a._native is not None and b._native is None
        assert (a.size, a.longest, a.total, a.tiles) == (b.size, b.longest, b.total, b.tiles)
        for _ in range(4):
            flat, cost = r.choice([0, 1, 2, 5, 128, 1000]), r.choice([0, 1, 2, 64])
            most = r.choice([None, 1, 16, 4096, 1 << 40])
            assert flat_needs_merge(torch.tensor(lens, dtype=torch.int32), flat, most, cost) \
                == flat_needs_merge(lens, flat, most, cost), (lens, flat, cost, most)


@pytest.mark.parametrize("kv,head_dim,hkv,group", [("fp16", 128, 8, 4), ("fp8_e5m2", 64, 2, 7), ("int8", 128, 8, 8)])
def test_plans_do_not_depend_on_how_lengths_arrive(kv, head_dim, hkv, group):
    for lens in _batches(9):
        forms = [lens, torch.tensor(lens, dtype=torch.int32), torch.tensor(lens, dtype=torch.int64)]
        if len(lens) > 1:  # a strided int32 view
            forms.append(torch.tensor([x for v in lens for x in (v, 5)], dtype=torch.int32)[::2])
        plans = [plan_launch(len(lens), 0, hkv, group, 256, 2, kv_dtype=kv, head_dim=head_dim, seq_lens=f) for f in forms]
        assert all(p == plans[0] for p in plans), lens


def test_argument_checks():
    lib = _abi.load()
    out = ctypes.c_int(0)
    stats = (ctypes.c_int64 * 3)()
    assert lib.pa_lens_stats(None, 2, stats) == _abi.PA_ERR_INVALID
    assert lib.pa_lens_stats(None, -1, stats) == _abi.PA_ERR_INVALID
    assert lib.pa_lens_stats(None, 0, None) == _abi.PA_ERR_INVALID
    assert lib.pa_lens_stats(None, 0, stats) == _abi.PA_OK and list(stats) == [0, 0, 0]
    assert lib.pa_flat_needs_merge(None, 2, 5, 1, 0, ctypes.byref(out)) == _abi.PA_ERR_INVALID
    assert lib.pa_flat_needs_merge(None, 0, 5, 1, -1, ctypes.byref(out)) == _abi.PA_ERR_INVALID
    assert lib.pa_flat_needs_merge(None, 0, 5, 1, 0, None) == _abi.PA_ERR_INVALID


def test_host_lengths_are_cpu_tensors():
    """A tensor without host memory (meta: its address reads as none given) is refused by flat
    launches, left out of unsplit ones, and never handed to the native pass."""
    from pagedattn.hip_decode import _check_host_lens, _host_lens_pointer

    ok, meta = torch.tensor([5, 6, 7], dtype=torch.int32), torch.empty(3, dtype=torch.int32, device="meta")
    _check_host_lens(ok, 3)
    assert _host_lens_pointer(ok, 3, 1, 0) == _host_lens_pointer(ok, 3, 1, 8) == ok.data_ptr()
    with pytest.raises(ValueError, match="contiguous int32 CPU tensor"):
        _check_host_lens(meta, 3)
    with pytest.raises(ValueError, match="contiguous int32 CPU tensor"):
        _host_lens_pointer(meta, 3, 1, 8)
    assert _host_lens_pointer(meta, 3, 1, 0) is None
    with pytest.raises(NotImplementedError):  # torch's own refusal to read it, not the library's
        _Lens(meta)
