"""mf_attention_plan_device: every tile of every column is planned exactly once
-- up to the context's end, since rows that share a position see past the
causal estimate -- and every partial slot is merged exactly once, over the
shapes the general planner takes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from memforge_amd import _native as nat


def _cover(items, merges, counts, q_lens, kv, hq, hkv, d):
    G = hq // hkv
    n_narrow, n_wide = int(counts[0]), int(counts[1])
    assert n_narrow % 4 == 0 and n_wide % 4 == 0 and items.shape[0] == n_narrow + n_wide
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    cover, slots = {}, {}
    for i, it in enumerate(items):
        s, h, c0, nct, kt0, kt1, slot, _, row0, rows, kvl, coop = (int(x) for x in it)
        if nct == 0:
            assert slot == -1
            continue
        assert (row0, rows, kvl) == (int(cu[s]), q_lens[s], kv[s])
        for c in range(c0, c0 + nct):
            cover.setdefault((s, h, c), []).append((kt0, kt1))
            if slot >= 0 and not (coop and i % 4):
                assert slot + c - c0 not in slots
                slots[slot + c - c0] = (s, h, c)
    for s, (q, n) in enumerate(zip(q_lens, kv)):
        for h in range(hkv):
            for c in range((q * G + 15) // 16 if n else 0):
                ranges = sorted(r for r in cover.pop((s, h, c)) if r[1] > r[0])
                assert ranges[0][0] == 0 and ranges[-1][1] == (n + 15) // 16
                assert all(a[1] == b[0] for a, b in zip(ranges, ranges[1:]))
    assert not cover
    named = {}
    for m in merges:
        s, h, c, n, slot0, stride = (int(x) for x in m[:6])
        for p in range(n):
            assert slots[slot0 + p * stride] == (s, h, c) and slot0 + p * stride not in named
            named[slot0 + p * stride] = True
    assert len(named) == len(slots)
    assert int(counts[3]) >= len(slots) * 16 * (max(d, 32) + 2)


@pytest.mark.parametrize("hq,hkv,d,dtype", [(15, 5, 64, torch.bfloat16), (40, 8, 128, torch.float16),
                                            (16, 4, 32, torch.bfloat16), (8, 2, 256, torch.bfloat16),
                                            (15, 5, 64, torch.float32), (8, 8, 16, torch.bfloat16)])
@pytest.mark.parametrize("cus", [1, 8, 256])
def test_device_plans_cover_every_tile_once(hq, hkv, d, dtype, cus):
    rng = np.random.default_rng(cus + d)
    shapes = [([1] * 9, [int(x) for x in rng.integers(1, 9000, 9)]), ([5] * 7, [int(x) for x in rng.integers(5, 3000, 7)]),
              ([1, 40, 7, 0, 130, 1, 3], [700, 2100, 7, 0, 5000, 1, 33]), ([512], [6656]), ([33], [33]),
              ([20, 300, 1024], [20, 2348, 1024])]
    for q_lens, kv in shapes:
        cu = np.concatenate([[0], np.cumsum(q_lens)]).tolist()
        made = nat.plan_attention_host(cu, kv, hq, hkv, d, dtype, num_cus=cus)
        _cover(*made, q_lens, kv, hq, hkv, d)


def test_device_plans_keep_wide_workgroups_shared_and_leave_full_grids_uncut():
    cu, kv = [0, 2048, 4096], [8000, 5000]
    items, merges, counts = nat.plan_attention_host(cu, kv, 40, 8, 128, torch.bfloat16, num_cus=256)
    assert merges.shape[0] == 0 and int((items[:, 5] - items[:, 4]).max()) == 500
    items, merges, counts = nat.plan_attention_host([0, 20, 31], [900, 3000], 15, 5, 64, torch.bfloat16, num_cus=256)
    assert int(counts[0]) == 0 and merges.shape[0] > 0  # few workgroups: ranges are cut
    for u in range(0, items.shape[0], 4):
        assert len({tuple(x[[0, 1, 4, 5]]) for x in items[u:u + 4]}) == 1


def test_device_plan_refuses_a_device_without_compute_units():
    a = np.array([0, 1], dtype=np.int32)
    counts = np.zeros(4, dtype=np.int64)
    assert nat.lib().mf_attention_plan_device(1, a.ctypes.data, a[1:].ctypes.data, 2, 1, 64, 2, 0, None, 0, None, 0,
                                              counts.ctypes.data) == -1


@pytest.mark.parametrize("heads,kv,single,cut", [
    ((15, 5, 64), [500], 4, False), ((15, 5, 64), [1152] * 64, 4, False),
    ((40, 8, 128), [1280] * 8, 4, False), ((40, 8, 128), [16000] * 2, 4, True),
])
def test_device_decode_plans_run_ranges_as_cooperative_units(heads, kv, single, cut):
    cu = list(range(len(kv) + 1))
    items, merges, counts = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16, num_cus=256)
    assert (merges.shape[0] > 0) == cut and (items[:, 11] == 1).all()
    if not cut:
        assert items.shape[0] == 4 * heads[1] * len(kv)
    _cover(items, merges, counts, [1] * len(kv), kv, *heads)
    short, none, counts = nat.plan_attention_host(cu, [16 * single] * len(kv), *heads, torch.bfloat16, num_cus=256)
    assert (short[:, 11] == 0).all() and int(counts[2]) == 0
    _cover(short, none, counts, [1] * len(kv), [16 * single] * len(kv), *heads)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads", [(15, 5, 64), (9, 3, 64), (40, 8, 128), (32, 32, 64)])
def test_device_decode_plans_reach_the_newest_key(heads, dtype):
    """Batches and contexts on both sides of every limit of the decode rule
    (pairs per compute unit, tiles of a single wave, rows that are cut): every
    range is planned to its last tile."""
    rng = np.random.default_rng(heads[0])
    for b in (1, 2, 7, 8, 32, 33, 40, 51, 52, 64, 85, 100, 102, 103, 170, 171, 256):
        for n in (1, 15, 17, 64, 65, 129, 256, 257, 500, 513, 1280, 1600, 2048):
            mixed = [int(x) for x in rng.integers(1, n + 1, b)]
            for kv in ([n] * b, mixed):
                made = nat.plan_attention_host(list(range(b + 1)), kv, *heads, dtype, num_cus=256)
                items = made[0]
                ends = np.zeros((b, heads[1]), dtype=np.int64)
                held = np.zeros((b, heads[1]), dtype=np.int64)
                live = items[items[:, 3] > 0]
                np.maximum.at(ends, (live[:, 0], live[:, 1]), live[:, 5])
                np.add.at(held, (live[:, 0], live[:, 1]), live[:, 5] - live[:, 4])
                tiles = (np.asarray(kv) + 15) // 16
                assert (ends == tiles[:, None]).all() and (held == tiles[:, None]).all(), (b, n)
        _cover(*made, [1] * b, kv, *heads)


def test_device_decode_plans_leave_full_grids_and_verify_rows_to_the_general_planner():
    for q, kv, heads in (([1] * 256, [4000] * 256, (40, 8, 128)), ([5] * 16, [1500] * 16, (15, 5, 64)),
                         ([1] * 9, [3000] * 9, (15, 5, 64))):
        cu = np.concatenate([[0], np.cumsum(q)]).tolist()
        a = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16, num_cus=256)
        b = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16)
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("cus,partition", [(0, 128), (0, 0), (256, 0)])
@pytest.mark.parametrize("hq,hkv,d,rows", [(40, 8, 128, 2), (15, 5, 64, 5)])
def test_single_column_items_fit_their_block_table_registers(cus, partition, hq, hkv, d, rows):
    """A wave holds the block-table entries of 128 tiles. The cut that gives a
    verify unit's last wave fewer tiles must leave the others no more than that,
    up to units of 512 tiles."""
    for tiles in (500, 506, 507, 509, 510, 511, 512, 1014, 1017, 1024):
        kv = [tiles * 16 - 3] * 32
        cu = [rows * i for i in range(33)]
        made = nat.plan_attention_host(cu, kv, hq, hkv, d, torch.bfloat16, partition, num_cus=cus)
        narrow = made[0][:int(made[2][0])]
        assert narrow.shape[0] and int((narrow[:, 5] - narrow[:, 4]).max()) <= nat.MAX_ITEM_TILES, tiles
        _cover(*made, [rows] * 32, kv, hq, hkv, d)


@pytest.mark.parametrize("heads,kv,kept", [
    ((9, 3, 64), [1400], True), ((15, 5, 64), [1400] * 4, True), ((40, 8, 128), [1772, 2171], True),  # short chains
    ((40, 8, 128), [1400] * 100, True),                                       # bytes, and an even grid
    ((40, 8, 128), [5000] * 33, False),                                       # bytes, 264 workgroups on 256 units
    ((15, 5, 64), [40 + 18 * i for i in range(64)], False), ((40, 8, 128), [8192, 12000, 20000, 24576], False),
])
def test_device_decode_rule_gives_way_where_the_general_plan_is_the_shorter(heads, kv, kept):
    cu = list(range(len(kv) + 1))
    a = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16, num_cus=256)
    b = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16)
    assert all(np.array_equal(x, y) for x, y in zip(a, b)) == kept
    _cover(*a, [1] * len(kv), kv, *heads)


@pytest.mark.parametrize("heads", [(40, 8, 128), (15, 5, 64)])
def test_merge_free_plans_hold_whole_ranges(heads):
    rng = np.random.default_rng(9)
    taken = 0
    for kv in ([int(x) for x in rng.integers(200, 3000, 64)], [8176, 1000, 1000], [8192] * 4, [1500] * 8, [300] * 20,
               [40 + 18 * i for i in range(64)], [9000] * 2):
        cu = list(range(len(kv) + 1))
        made = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16, num_cus=256, merge_free=True)
        _cover(*made, [1] * len(kv), kv, *heads)
        general = nat.plan_attention_host(cu, kv, *heads, torch.bfloat16)
        if not all(np.array_equal(x, y) for x, y in zip(made, general)):
            assert made[1].shape[0] == 0 and max(kv) <= 8192
            taken += 1
    assert taken >= (3 if heads[2] == 128 else 1)


@pytest.mark.parametrize("seqs,keys,rows,parts", [
    (3, 330, 8, 1),                  # few workgroups, 21 tiles: whole
    (3, 450, 8, 4), (16, 440, 8, 4),  # few workgroups: ranges of about 8 tiles
    (40, 490, 8, 1),                 # more workgroups, 31 tiles: whole
    (40, 1000, 8, 3),                # more, and enough work for two workgroups a compute unit
])
def test_short_wide_launches_are_cut_finely_or_not_at_all(seqs, keys, rows, parts):
    cu, kv = [rows * i for i in range(seqs + 1)], [keys] * seqs
    made = nat.plan_attention_host(cu, kv, 15, 5, 64, torch.bfloat16, num_cus=256)
    _cover(*made, [rows] * seqs, kv, 15, 5, 64)
    assert int(made[2][0]) == 0 and int(made[2][1]) == 4 * 5 * seqs * parts
