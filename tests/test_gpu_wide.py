"""Workgroup-shared wide items (attn_wide_body) where they can go wrong: stage
and block edges, ranges past one block-table refill (64 tiles), the boundary
between pool and new rows, rows behind a row map, padding columns and waves,
rows that share a position, NaN past the context, and both layouts -- against
the float64 oracle. The tolerance is the attention tests' (bf16 2e-2, fp16
4e-3 max-abs on N(0,1) values: 2^-8 and 2^-11 relative on P and the output)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from memforge_amd import _native as nat
from memforge_amd.models.paged_attention import PagedAttention, PagedKVCache
from oracle import attention as oatt
from tests.gpu_helpers import pad_tables, random_tables, to_np64

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3}


def _plan(cu, kv, hq, hkv, d, dtype, dev, cus):
    items, merges, counts = nat.plan_attention_host(cu, kv, hq, hkv, d, dtype, num_cus=cus)
    di, dm = nat.upload(nat.plan_upload_parts(items, merges), dev)
    return nat.plan_from_parts(items, merges, counts, di, dm)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(6, 2, 32), (15, 5, 64), (10, 2, 128)])
@pytest.mark.parametrize("cus", [1, 256])  # ranges uncut / cut for a whole device
@pytest.mark.parametrize("form", ["write", "inflight", "pool"])
def test_wide_items_match_the_oracle(dtype, hq, hkv, d, cus, form):
    _against_the_oracle(dtype, hq, hkv, d, cus, form, 16)


@pytest.mark.parametrize("bs,dtype", [(1, torch.bfloat16), (8, torch.float16), (12, torch.bfloat16),
                                      (32, torch.float16), (48, torch.bfloat16)])
@pytest.mark.parametrize("hq,hkv,d", [(6, 2, 32), (15, 5, 64), (10, 2, 128)])
@pytest.mark.parametrize("cus", [0, 1, 256])  # 0: the general planner
@pytest.mark.parametrize("form", ["inflight", "pool"])
def test_wide_items_on_other_block_sizes_match_the_oracle(bs, dtype, hq, hkv, d, cus, form):
    """Blocks smaller and larger than a tile, a stage and not a power of two."""
    _against_the_oracle(dtype, hq, hkv, d, cus, form, bs)


def _against_the_oracle(dtype, hq, hkv, d, cus, form, bs):
    dev = torch.device("cuda:0")
    gen = torch.Generator().manual_seed(d + cus)
    # (prior keys, new rows): one tile of columns more than narrow, uneven
    # boundaries, a fresh prompt, more than 128 tiles of pool, one row short of
    # and past a stage, rows only just wide
    runs = [(0, 64), (2075, 37), (13, 130), (64, 63), (129, 65), (31, 17), (1040, 6)]
    kv = [p + n for p, n in runs]
    nblocks = sum((k + bs - 1) // bs for k in kv) + 2
    tables = random_tables(gen, nblocks, kv, bs)
    kp = torch.randn((nblocks, bs, hkv, d), generator=gen).to(dtype)
    vp = torch.randn((nblocks, bs, hkv, d), generator=gen).to(dtype)
    T = sum(n for _, n in runs)
    q = torch.randn((T, hq, d), generator=gen).to(dtype)
    nk = torch.randn((T, hkv, d), generator=gen).to(dtype)
    nv = torch.randn((T, hkv, d), generator=gen).to(dtype)
    cu = np.concatenate([[0], np.cumsum([n for _, n in runs])]).tolist()
    seq_ids = [i for i, (_, n) in enumerate(runs) for _ in range(n)]
    positions = [p + j for p, n in runs for j in range(n)]
    slots = [tables[s][p // bs] * bs + p % bs for s, p in zip(seq_ids, positions)]
    full_k, full_v = kp.clone(), vp.clone()
    full_k.view(-1, hkv, d)[slots] = nk
    full_v.view(-1, hkv, d)[slots] = nv
    want = oatt.varlen_attention(to_np64(q.permute(1, 0, 2)), to_np64(full_k), to_np64(full_v), tables, seq_ids,
                                 positions, bs)
    # slots past each context hold NaN
    src_k, src_v = (full_k, full_v) if form == "pool" else (kp.clone(), vp.clone())
    for t, k in zip(tables, kv):
        if k % bs:
            src_k[t[-1], k % bs:] = float("nan")
            src_v[t[-1], k % bs:] = float("nan")
    dk, dv = src_k.to(dev), src_v.to(dev)
    pool = nat.PoolView.from_bshd(dk, dv)
    out = torch.full((T, hq, d), float("nan"), dtype=dtype, device=dev)
    plan = _plan(cu, kv, hq, hkv, d, dtype, dev, cus)
    assert plan.n_wide > 0
    meta = (pad_tables(tables, dev), torch.tensor(cu, dtype=torch.int32, device=dev),
            torch.tensor(kv, dtype=torch.int32, device=dev))
    pos_t = torch.tensor(positions, dtype=torch.int64, device=dev)
    scale = 1.0 / float(np.sqrt(d))
    if form == "write":
        nat.paged_attention_kv_write(q.to(dev), out, pool, *meta, pos_t, plan, scale, hkv, nk.to(dev), nv.to(dev),
                                     torch.tensor(slots, dtype=torch.int64, device=dev))
        assert torch.equal(dk.cpu().view(-1, hkv, d)[slots], nk) and torch.equal(dv.cpu().view(-1, hkv, d)[slots], nv)
    elif form == "inflight":
        # physical rows in another order, reached through the row map
        perm = torch.randperm(T, generator=gen)
        inv = torch.empty_like(perm)
        inv[perm] = torch.arange(T)
        nat.paged_attention(q[inv].to(dev), out, pool, *meta, pos_t.cpu()[inv].to(dev), plan, scale, hkv,
                            row_map=perm.to(torch.int32).to(dev),
                            pool_lens=torch.tensor([p for p, _ in runs], dtype=torch.int32, device=dev),
                            new_k_rows=nk[inv].to(dev), new_v_rows=nv[inv].to(dev))
        out = out[perm.to(dev)]
    else:
        nat.paged_attention(q.to(dev), out, pool, *meta, pos_t, plan, scale, hkv)
    err = np.abs(to_np64(out.permute(1, 0, 2)) - want)
    assert err.max() <= TOL[dtype], err.max()


@pytest.mark.parametrize("q_len,ctx", [(33, 300), (70, 2200), (130, 65)])
def test_rows_that_share_a_position_see_the_whole_context(q_len, ctx):
    """The operator's queries are not causal: every row of a wide item reads
    every key, past the planner's causal estimate."""
    gen = torch.Generator().manual_seed(ctx)
    h, d, bs = 4, 64, 16
    blocks = (ctx + bs - 1) // bs
    cache = PagedKVCache(blocks + 1, bs, h, d, dtype=torch.bfloat16)
    table = torch.randperm(blocks + 1, generator=gen)[:blocks].tolist()
    k = torch.randn((1, h, ctx, d), generator=gen).to(torch.bfloat16)
    v = torch.randn((1, h, ctx, d), generator=gen).to(torch.bfloat16)
    q = torch.randn((1, h, q_len, d), generator=gen).to(torch.bfloat16)
    cache.write_kv(k.cuda(), v.cuda(), table, 0)
    got = PagedAttention()(q.cuda(), cache, table, ctx)
    want = oatt.paged_operator(to_np64(q), to_np64(cache.key_cache), to_np64(cache.value_cache), table, ctx)
    assert np.abs(to_np64(got) - want).max() <= TOL[torch.bfloat16]
