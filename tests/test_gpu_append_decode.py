"""Append, decode and the lengths' advance in one call: the advance rides on the
combine launch (or on one of its own after the per-sequence kernel), for every
kind of launch and both length types, eager and replayed from a graph."""

from __future__ import annotations

import pytest
import torch

import mxflashattn_amd as mx
from mxflashattn_amd import native
from mxflashattn_amd.workloads import make_paged_batch
from oracle import reference_port

TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}

pytestmark = pytest.mark.gpu


# (tokens, GQ, table width in pages): the split kernel, several column groups,
# two launches of them (64 columns at head dim 128), the per-sequence kernel.
@pytest.mark.parametrize("ql,gq,width", [(1, 4, 100), (8, 4, 100), (16, 4, 100), (1, 2, 16),
                                         (3, 2, 16)])
@pytest.mark.parametrize("lengths", [torch.int32, torch.int64], ids=["int32", "int64"])
def test_lengths_advance_with_the_decode(device, taken, ql, gq, width, lengths):
    batch = 70 if width == 16 else 5
    start = torch.arange(batch) % 7 * 33
    b = make_paged_batch(batch, 2 * gq, 2, 128, torch.bfloat16, start + 3 * ql, q_len=ql,
                         block_table_width=width, seed=ql)
    kc, vc, lens = b.k_cache.to(device), b.v_cache.to(device), start.to(device, lengths)
    ref_k, ref_v, ref_lens = b.k_cache.clone(), b.v_cache.clone(), start.clone()
    g = torch.Generator().manual_seed(width + ql)
    for step in range(3):
        q, k, v = (torch.randn(batch, ql, h, 128, generator=g).to(torch.bfloat16)
                   for h in (2 * gq, 2, 2))
        taken.clear()
        want = reference_port.attention_kvcache(
            q.float(), ref_k, ref_v, cache_seqlens=ref_lens, block_table=b.block_table, k=k, v=v,
            softmax_scale=b.scale, causal=True).float()
        out = mx.flash_attn_with_kvcache(q.to(device), kc, vc, k=k.to(device), v=v.to(device),
                                         cache_seqlens=lens, block_table=b.block_table.to(device),
                                         softmax_scale=b.scale, causal=True)
        assert (out.float().cpu() - want).abs().max().item() <= TOL[torch.bfloat16], step
        assert lens.cpu().tolist() == (start + (step + 1) * ql).tolist()
        # int64 lengths take the binding, and torch adds to them.
        assert taken == (["append_kv", "decode_tokens"] if lengths == torch.int32 else [])
        assert torch.equal(kc.cpu(), ref_k) and torch.equal(vc.cpu(), ref_v)


def test_lengths_advance_on_every_replay(device, taken):
    b = make_paged_batch(4, 16, 4, 128, torch.bfloat16, torch.tensor([300, 5, 90, 64]), q_len=2,
                         block_table_width=40, seed=3).to(device)
    k, v = (torch.randn(4, 2, 4, 128, device=device).to(torch.bfloat16) for _ in range(2))
    start = torch.tensor([200, 0, 77, 40], dtype=torch.int32, device=device)
    lens, stream = start.clone(), torch.cuda.Stream(device)
    out = torch.empty_like(b.q)

    def call():
        return mx.flash_attn_with_kvcache(b.q, b.k_cache, b.v_cache, k=k, v=v, cache_seqlens=lens,
                                          block_table=b.block_table, causal=True, out=out)

    eager = []
    with torch.cuda.stream(stream):
        for _ in range(4):
            eager.append(call().clone())
        lens.copy_(start)
        call()
    torch.cuda.synchronize()
    lens.copy_(start)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    taken.clear()
    with torch.cuda.graph(graph, stream=stream):
        call()
    assert taken == ["append_kv", "decode_tokens"]
    for i, want in enumerate(eager):
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        assert lens.tolist() == (start + 2 * (i + 1)).tolist()
        torch.ones(1 << 20, device=device).sum().item()  # eager work between replays


# 512 heads of 4096 elements: 2^18 fragments a row. 8128 rows are the most that
# the 32-bit index arithmetic takes; one more, and past 2^31, take the 64-bit one.
@pytest.mark.parametrize("rows", [8128, 8129, 8200])
@pytest.mark.parametrize("kind", ["slots", "fp8", "table"])
def test_appends_past_32_bit_indexes(device, taken, kind, rows):
    g = torch.Generator(device=device).manual_seed(rows)
    dt = torch.float8_e4m3fn if kind == "fp8" else torch.bfloat16
    base = torch.randn(512 * 4096 + 8 * rows, generator=g, device=device).to(torch.bfloat16)
    flat = base.as_strided((rows, 512, 4096), (8, 4096, 1))  # every row another window
    kc, vc = (torch.zeros(2, 2, 512, 4096, device=device).to(dt) for _ in range(2))
    if kind == "table":  # one sequence; all but the last two positions lie before 0
        lens = torch.tensor([2 - rows], dtype=torch.int32, device=device)
        table = torch.tensor([[1]], dtype=torch.int32, device=device)
        native.append_kv(flat[None], flat[None], kc, vc, table, lens)
        where = {2: rows - 2, 3: rows - 1}
    else:
        where = {1: 0, 2: rows // 2, 0: rows - 1}
        slots = torch.full((rows,), -1, dtype=torch.int64, device=device)
        for slot, row in where.items():
            slots[row] = slot
        scale = torch.full((1,), 0.5, device=device) if kind == "fp8" else None
        native.reshape_and_cache(flat, flat, kc, vc, slots, k_scale=scale, v_scale=scale)
    assert len(taken) == 1
    for cache in (kc, vc):
        got = cache.flatten(0, 1)
        for slot in range(4):
            want = torch.zeros(512, 4096, device=device).to(dt)
            if slot in where:
                want = flat[where[slot]]
                if kind == "fp8":
                    want = (want.float() / 0.5).clamp(-448, 448).to(dt)
            assert torch.equal(got[slot].view(torch.uint8), want.contiguous().view(torch.uint8))


def test_a_slot_past_32_bits(device, taken):
    # Pages that share their rows: 2^28 of 16 tokens without the memory of them.
    kc, vc = (torch.zeros(1, 16, 1, 64, device=device).to(torch.bfloat16).expand(2 ** 28, -1, -1, -1)
              for _ in range(2))
    k = torch.randn(2, 1, 64, device=device).to(torch.bfloat16)
    slots = torch.tensor([2 ** 31 + 5, 2 ** 32 + 7], device=device)  # the second: no such page
    native.reshape_and_cache(k, k, kc, vc, slots)
    assert taken == ["reshape_and_cache"]
    want = torch.zeros(16, 1, 64, dtype=torch.bfloat16, device=device)
    want[5] = k[0]
    assert torch.equal(kc[0], want) and torch.equal(vc[0], want)
