"""Decode steps planned for a device (mf_attention_plan_device) through the
entry points that use such plans, against the float64 oracle and, for whole
graphed steps, plain transformers attention."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from memforge_amd import _native as nat
from memforge_amd.kernels.varlen_attention import paged_attention_varlen
from oracle import attention as oatt
from tests.gpu_helpers import pad_tables, random_tables, to_np64
from tests.tiny_models import tiny_llama

pytestmark = pytest.mark.gpu

# the attention tests' tolerances on N(0,1) values: 2^-8 and 2^-11 relative on
# P and the output, and fp32 sums
TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}


def _decode_case(batch, keys, hq, hkv, d, dtype):
    gen = torch.Generator().manual_seed(batch + keys)
    kv = [keys] * batch
    blocks = batch * ((keys + 15) // 16) + 3
    tables = random_tables(gen, blocks, kv, 16)
    kp = torch.randn((blocks, 16, hkv, d), generator=gen).to(dtype)
    vp = torch.randn((blocks, 16, hkv, d), generator=gen).to(dtype)
    q = torch.randn((batch, hq, d), generator=gen).to(dtype)
    want = oatt.varlen_attention(to_np64(q.permute(1, 0, 2)), to_np64(kp), to_np64(vp), tables, list(range(batch)),
                                 [keys - 1] * batch, 16)
    return kv, tables, kp, vp, q, want


# More (sequence, kv head) pairs than compute units and contexts of more tiles
# than the general partition gives one wave.
SHORT = [(64, 256, 15, 5, 64, torch.bfloat16), (100, 250, 9, 3, 64, torch.float32),
         (40, 256, 40, 8, 128, torch.float16)]


@pytest.mark.parametrize("batch,keys,hq,hkv,d,dtype", SHORT)
def test_batched_decodes_of_short_contexts_attend_every_key(device, batch, keys, hq, hkv, d, dtype):
    kv, tables, kp, vp, q, want = _decode_case(batch, keys, hq, hkv, d, dtype)
    dk, dv, dq = kp.to(device), vp.to(device), q.to(device)
    got = paged_attention_varlen(dq.permute(1, 0, 2).unsqueeze(0), dk.unsqueeze(0), dv.unsqueeze(0), 0, tables,
                                 list(range(batch)), [keys - 1] * batch, 16)
    assert np.abs(to_np64(got[0]) - want).max() <= TOL[dtype]
    # the same step with its newest rows written in flight
    slots = [t[(keys - 1) // 16] * 16 + (keys - 1) % 16 for t in tables]
    new_k, new_v = dk.view(-1, hkv, d)[slots].clone(), dv.view(-1, hkv, d)[slots].clone()
    dk.view(-1, hkv, d)[slots] = float("nan")
    dv.view(-1, hkv, d)[slots] = float("nan")
    out = torch.full_like(dq, float("nan"))
    plan = nat.plan_attention(list(range(batch + 1)), kv, hq, hkv, d, dtype, device)
    nat.paged_attention_kv_write(
        dq, out, nat.PoolView.from_bshd(dk, dv), pad_tables(tables, device),
        torch.arange(batch + 1, dtype=torch.int32, device=device), torch.tensor(kv, dtype=torch.int32, device=device),
        torch.full((batch,), keys - 1, dtype=torch.int64, device=device), plan, d ** -0.5, hkv, new_k, new_v,
        torch.tensor(slots, dtype=torch.int64, device=device))
    assert np.abs(to_np64(out.permute(1, 0, 2)) - want).max() <= TOL[dtype]


def test_graphed_decodes_of_short_contexts_attend_every_key(device):
    """A whole graphed step of 12 sequences of 256 keys, 32 kv heads, against
    transformers' own attention over the same cached keys."""
    from transformers.cache_utils import DynamicCache

    from memforge_amd.runtime.graphed_paged_decode import GraphedPagedDecoder
    from memforge_amd.runtime.kv_pool import ModelKVSpec, PagedKVPool

    batch, ctx, layers = 12, 255, 2
    model = tiny_llama(num_layers=layers, heads=32, kv_heads=32, head_dim=16)
    pool = PagedKVPool(ModelKVSpec.from_config(model.config, torch.float32, "cuda:0"), batch * 16 + 4, 16)
    gen = torch.Generator().manual_seed(3)
    pool.key_pool.copy_(torch.randn(pool.key_pool.shape, generator=gen).to(device))
    pool.value_pool.copy_(torch.randn(pool.value_pool.shape, generator=gen).to(device))
    tables = random_tables(gen, batch * 16 + 4, [ctx + 1] * batch, 16)
    tokens = [7 + 3 * i for i in range(batch)]
    cache = DynamicCache()
    slots = torch.tensor([[t[p // 16] * 16 + p % 16 for p in range(ctx)] for t in tables], device=device)
    for i in range(layers):
        k, v = (p[i].reshape(-1, 32, 16)[slots].permute(0, 2, 1, 3).contiguous()
                for p in (pool.key_pool, pool.value_pool))
        cache.update(k, v, i)
    with torch.no_grad():
        want = model(input_ids=torch.tensor(tokens, device=device).view(batch, 1),
                     position_ids=torch.full((batch, 1), ctx, device=device), past_key_values=cache,
                     use_cache=True).logits[:, -1]
    dec = GraphedPagedDecoder(model, pool, max_batch=16, max_model_len=300)
    for _ in range(3):  # the same step again: every replay rewrites the same rows
        torch.testing.assert_close(dec.step(tokens, [ctx] * batch, tables), want, atol=2e-5, rtol=1e-4)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,lo,hi,hq,hkv,d", [(8, 1500, 1501, 40, 8, 128), (16, 500, 4000, 40, 8, 128),
                                                  (3, 9000, 12000, 8, 2, 256)])
def test_cut_decode_ranges_round_their_output_once(device, batch, lo, hi, hq, hkv, d, dtype, fused):
    """A device plan's cut ranges, against one whole unit's accuracy. All scores
    are 0, so every weight is 1, every product exact, and each output element is
    the mean of its values: fp32 sums of n values of N(0,1) are off by about
    2^-24 sqrt(n) on sums of about sqrt(n), far below the rounding step of the
    16-bit output, and all but a few elements (those within that error of a
    rounding boundary: under 1% in bf16, 5% in fp16) are the rounded mean.
    Partial outputs rounded to 16 bits before the merge get a third wrong."""
    rng = np.random.default_rng(batch)
    gen = torch.Generator().manual_seed(batch)
    kv = [int(x) for x in rng.integers(lo, hi, batch)]
    blocks = sum((n + 15) // 16 for n in kv) + 3
    tables = random_tables(gen, blocks, kv, 16)
    kp = torch.randn((blocks, 16, hkv, d), generator=gen).to(dtype).to(device)
    vp = torch.randn((blocks, 16, hkv, d), generator=gen).to(dtype).to(device)
    q = torch.zeros((batch, hq, d), dtype=dtype, device=device)
    plan = nat.plan_attention(list(range(batch + 1)), kv, hq, hkv, d, dtype, device)
    assert plan.n_merges > 0
    out = torch.full_like(q, float("nan"))
    nat.paged_attention(q, out, nat.PoolView.from_bshd(kp, vp), pad_tables(tables, device),
                        torch.arange(batch + 1, dtype=torch.int32, device=device),
                        torch.tensor(kv, dtype=torch.int32, device=device),
                        torch.tensor(kv, dtype=torch.int64, device=device) - 1, plan, d ** -0.5, hkv,
                        fused_merge=fused)
    wrong = 0
    for i, (t, n) in enumerate(zip(tables, kv)):
        mean = vp[t].reshape(-1, hkv, d)[:n].double().mean(0).to(dtype)
        wrong += int((out[i].view(hkv, hq // hkv, d) != mean[:, None]).sum())
    share = wrong / out.numel()
    assert share <= (0.01 if dtype == torch.bfloat16 else 0.05), share


def test_graphed_decoder_plans_a_merge_free_step_once(device, monkeypatch):
    """Ranges that a device plan would cut (256-byte rows and more, over 80
    tiles): the merge-free decoder asks once, for whole ranges, and runs them as
    cooperative units; against transformers' attention."""
    from transformers.cache_utils import DynamicCache

    from memforge_amd.runtime.graphed_paged_decode import GraphedPagedDecoder
    from memforge_amd.runtime.kv_pool import ModelKVSpec, PagedKVPool

    ctx, tokens = [2100, 1000, 999], [9, 12, 40]
    model = tiny_llama(num_layers=1, heads=4, kv_heads=2, head_dim=128)
    blocks = sum((c + 16) // 16 for c in ctx) + 2
    pool = PagedKVPool(ModelKVSpec.from_config(model.config, torch.float32, "cuda:0"), blocks, 16)
    gen = torch.Generator().manual_seed(4)
    pool.key_pool.copy_(torch.randn(pool.key_pool.shape, generator=gen).to(device))
    pool.value_pool.copy_(torch.randn(pool.value_pool.shape, generator=gen).to(device))
    tables = random_tables(gen, blocks, [c + 1 for c in ctx], 16)
    want = []
    for t, c, tok in zip(tables, ctx, tokens):
        slots = torch.tensor([t[p // 16] * 16 + p % 16 for p in range(c)], device=device)
        cache = DynamicCache()
        cache.update(*(p[0].reshape(-1, 2, 128)[slots].transpose(0, 1).unsqueeze(0).contiguous()
                       for p in (pool.key_pool, pool.value_pool)), 0)
        with torch.no_grad():
            want.append(model(input_ids=torch.tensor([[tok]], device=device),
                              position_ids=torch.tensor([[c]], device=device), past_key_values=cache,
                              use_cache=True).logits[0, -1])
    made = []
    plan = nat.plan_attention_host
    monkeypatch.setattr(nat, "plan_attention_host", lambda *a, **kw: made.append(plan(*a, **kw)) or made[-1])
    dec = GraphedPagedDecoder(model, pool, max_batch=4, max_model_len=2200)
    assert dec.merge_free
    for _ in range(3):
        torch.testing.assert_close(dec.step(tokens, ctx, tables), torch.stack(want), atol=2e-5, rtol=1e-4)
    assert len(made) == 3 and all((items[:, 11] == 1).all() and counts[2] == 0 for items, _, counts in made)
