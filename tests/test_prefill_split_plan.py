"""Host-side split prefill plan (pl_prefill_split_plan): every row item's kv
tiles are covered once, cut ranges are listed for the merge, and what
pl_prefill_plan refuses is refused alike.  Reads host tables only."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from pagelora_amd import _lib

ROWS, TILE, PART_FLOATS = 128, 64, 128 * 130


def _plan(qo_lens, kv_lens, hq, hkv, ps, causal=True):
    lib = _lib.load()
    pages = [-(-n // ps) for n in kv_lens]
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    kv = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    last = np.array([n - ps * (p - 1) for n, p in zip(kv_lens, pages)], dtype=np.int32)
    n, m, ws = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t()
    args = (qo.ctypes.data, kv.ctypes.data, last.ctypes.data, len(kv_lens), hq, hkv, ps, int(causal))
    counts = (ctypes.byref(n), ctypes.byref(m), ctypes.byref(ws))
    _lib.check(lib.pl_prefill_split_plan(*args, None, 0, *counts), "pl_prefill_split_plan")
    records = np.zeros((max(1, n.value + m.value), 8), dtype=np.int32)
    _lib.check(lib.pl_prefill_split_plan(*args, records.ctypes.data, n.value + m.value, *counts),
               "pl_prefill_split_plan")
    return records[: n.value], records[n.value: n.value + m.value], ws.value


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv,qo_lens,kv_lens,ps", [
    (32, 8, [77], [32077], 16), (32, 32, [2119], [2119], 16), (28, 4, [1, 0, 40], [9000, 3, 40], 4),
    (8, 8, [300, 7], [300, 20000], 64), (4, 1, [5], [5], 12)])
def test_tiles_covered_once(hq, hkv, qo_lens, kv_lens, ps, causal):
    items, merges, ws = _plan(qo_lens, kv_lens, hq, hkv, ps, causal)
    g = hq // hkv
    want = {}
    for r, (n, kv) in enumerate(zip(qo_lens, kv_lens)):
        for r0 in range(0, n * g, ROWS):
            pos = kv - n + (min(r0 + ROWS, n * g) - 1) // g if causal else kv - 1
            want[r, r0] = pos // TILE + 1
    got, slots = {}, {}
    for r, r0, t0, t1, slot, part, parts, _ in items.tolist():
        assert t0 < t1 and (slot < 0) == (parts == 1)
        got.setdefault((r, r0), []).append((t0, t1))
        if slot >= 0:
            slots.setdefault((r, r0), []).append(slot + part)
    for key, ranges in got.items():
        ranges.sort()
        assert ranges[0][0] == 0 and ranges[-1][1] == want[key]
        assert all(a[1] == b[0] for a, b in zip(ranges, ranges[1:]))
    assert set(got) == set(want)
    lengths = [t1 - t0 for _, _, t0, t1, *_ in items.tolist()]
    assert lengths == sorted(lengths, reverse=True)
    # each cut item has one merge over its own slots, and the workspace holds all of them
    assert {(m[0], m[1]): list(range(m[4], m[4] + m[6])) for m in merges.tolist()} == \
        {k: sorted(v) for k, v in slots.items()}
    used = sorted(s for v in slots.values() for s in v)
    assert used == list(range(len(used))) and ws == len(used) * hkv * PART_FLOATS * 4


def test_refusals():
    with pytest.raises(ValueError, match="exceeds kv_len"):
        _plan([9], [8], 2, 2, 4)
    with pytest.raises(ValueError, match="multiple of 4"):
        _plan([1], [8], 2, 2, 2)
    with pytest.raises(ValueError, match="multiple of num_kv_heads"):
        _plan([1], [8], 3, 2, 4)
