"""The work that programs have this package do, as cases for timing.

Decode attention over a KV cache through the public entry points, from one
request to hundreds, short and long contexts, paged, dense and packed caches,
16-bit and fp8, one query token and several, and the cache writes that go with
it. ``listed()`` names the cases, ``draw(rng)`` gives others of the same
ranges; ``prepare`` makes one case's inputs, ``run`` is one pass of a user's
program, ``exact`` the same outputs in 64 bits from plain torch.
"""

import math
import types

import torch

import mxflashattn_amd as mx
from mxflashattn_amd.integrations.vllm.decode_step import DecodeMetadata
from mxflashattn_amd.integrations.vllm.decoder_adapter import forward_decode, kv_cache_update

DEVICE = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
# K/V bytes a drawn case reads or writes at most (config 2's 604 MB is the
# most a listed case reads).
MOST_BYTES = 560e6


def _case(name, kind, batch, q_heads, kv_heads, head_dim, dtype, lo, hi, **more):
    """One case. lo, hi: sequence lengths (uniform integers; ``spread``
    "lognormal": median 1024, clipped to [lo, hi]). page_size; capacity: keys
    a block-table row has room for (0: the longest sequence's)."""
    case = dict(kind=kind, batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                dtype=dtype, lo=lo, hi=hi, page_size=16, capacity=0, q_len=1, fp8=False,
                window=-1, softcap=0.0, sinks=False, alibi=False, spread="uniform")
    case.update(more)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest call: four short requests of a small model. Latency.
        _case("few_short_d64", "paged", 4, 8, 2, 64, "f16", 1, 512, capacity=512),
        # One user's chat turn on the Qwen3-4B shape, the table sized for the
        # model's context: latency, and a grid with little work for 256 CUs.
        _case("one_request_d128", "paged", 1, 32, 8, 128, "bf16", 2049, 2049, capacity=8192),
        # Many short requests in flight (BASELINE's high-batch shape).
        _case("many_short_gq2_d64", "paged", 128, 16, 8, 64, "f16", 1, 512),
        # The ordinary serving batch, and the headline shape.
        _case("serving_gq4_d128", "paged", 32, 32, 8, 128, "bf16", 1024, 8192),
        # The same lengths on the model with the smallest cache per token.
        _case("serving_gq8_d64", "paged", 32, 32, 4, 64, "bf16", 1024, 8192, page_size=64),
        # Long contexts, all equal.
        _case("long_gq8_d128", "paged", 16, 32, 4, 128, "bf16", 16384, 16384),
        # Speculative decoding: eight tokens per request appended and verified
        # in one causal call.
        _case("verify8_gq4_d128", "verify", 32, 32, 8, 128, "bf16", 1024, 8192, q_len=8),
        # Packed keys, one query token per sequence (the varlen entry point).
        _case("packed_gq4_d128", "varlen", 32, 32, 8, 128, "bf16", 1024, 8192),
        # A dense cache of an odd length, as a plain generation loop grows it.
        _case("dense_odd_gq2_d128", "dense", 16, 16, 8, 128, "f16", 4095, 4095),
        # One layer of a vLLM decode step with an fp8 cache: the token's K/V
        # written, then attention over lengths spread as real prompts are.
        _case("vllm_layer_fp8_d128", "layer", 128, 32, 8, 128, "bf16", 16, 8192, fp8=True,
              spread="lognormal"),
        # A local layer: sliding window and soft-capped logits, head dim 256.
        _case("window_softcap_d256", "options", 32, 16, 8, 256, "bf16", 1024, 8192, window=1023,
              softcap=50.0),
        # The cache write of a prefill: 8192 tokens' K and V to their slots.
        _case("prefill_write_d128", "write", 1, 32, 8, 128, "bf16", 8192, 8192),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["paged", "paged", "paged", "verify", "varlen", "dense", "layer", "options",
                       "write"])
    head_dim = rng.choice([64, 128])
    kv_heads = rng.choice([1, 2, 4, 5, 8, 16])
    gq = rng.choice([1, 2, 3, 4, 5, 8, 16])
    dtype = rng.choice(["f16", "bf16"])
    batch = _log(rng, 1, 200)
    more = {"page_size": rng.choice([16, 16, 32, 64, 256])}
    if kind == "verify":
        gq = rng.choice([2, 4, 8])
        more["q_len"] = rng.randint(2, 64 // gq if gq > 4 else 12)
    elif kind == "options":
        head_dim = rng.choice([64, 128, 256])
        more["fp8"] = rng.random() < 0.3
        if rng.random() < 0.5:
            more["window"] = _log(rng, 64, 4096)
        more["sinks"] = rng.random() < 0.4
        more["alibi"] = rng.random() < 0.2
        more["softcap"] = rng.choice([0.0, 30.0])
    elif kind == "layer":
        more["fp8"] = rng.random() < 0.5
    row = 2 * kv_heads * head_dim * (1 if more.get("fp8") else 2)  # K and V bytes of a token
    if kind == "write":
        batch = 1
    most = max(64, int(min(16384, MOST_BYTES / (row * batch))))
    hi = _log(rng, 256 if kind == "write" else 33, most)
    if kind in ("dense", "write"):
        lo = hi = hi | 1 if rng.random() < 0.7 else hi
    else:
        lo = rng.choice([1, max(1, hi // 8), hi])
    if kind in ("paged", "layer", "options") and rng.random() < 0.5:
        more["capacity"] = min(16384, 2 * hi)
    return _case(None, kind, batch, kv_heads * gq, kv_heads, head_dim, dtype, lo, hi, **more)


# ---------------------------------------------------------------------------
# Inputs


def _lengths(case):
    """Sequence lengths (the tokens being decoded included): a fixed draw per
    shape, so that every seed's pass does the same work on other values."""
    g = torch.Generator().manual_seed(20261007 + case["batch"])
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    if case["spread"] == "lognormal":
        z = torch.randn(b, generator=g, dtype=torch.float64)
        lens = torch.exp(math.log(1024.0) + z).round().clamp(lo, hi).to(torch.int64)
    else:
        lens = torch.randint(lo, hi + 1, (b,), generator=g)
    return lens.clamp(min=case["q_len"])


def _normal(g, *shape, dtype):
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)


def _pages(case, lens, seed):
    """(pages in the pool, block table int32 [B, W] on the host): every
    sequence owns distinct pages from a shuffled pool a quarter larger."""
    ps = case["page_size"]
    need = (lens + ps - 1) // ps
    total = int(need.sum())
    pool = math.ceil(1.25 * total)
    width = max(int(need.max()), -(-case["capacity"] // ps))
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    table = torch.zeros(case["batch"], width, dtype=torch.int32)
    live = torch.arange(width)[None, :] < need[:, None]
    table[live] = perm[:total]
    return pool, table


def prepare(case, seed):
    """What the program holds before the call, on the GPU."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dt, hd, hkv, hq = DTYPES[case["dtype"]], case["head_dim"], case["kv_heads"], case["q_heads"]
    b, ql, kind = case["batch"], case["q_len"], case["kind"]
    lens = _lengths(case)
    s = types.SimpleNamespace(case=case, kind=kind, lens=lens, scale=hd ** -0.5)
    if kind == "write":
        n = case["hi"]
        pool = math.ceil(1.25 * n / case["page_size"])
        s.key, s.value = (_normal(g, n, hkv, hd, dtype=dt) for _ in range(2))
        s.kc, s.vc = (torch.zeros(pool, case["page_size"], hkv, hd, device=DEVICE, dtype=dt)
                      for _ in range(2))
        order = torch.randperm(pool, generator=torch.Generator().manual_seed(seed))
        slots = (order[:, None] * case["page_size"] + torch.arange(case["page_size"])).flatten()
        s.slots = slots[:n].to(DEVICE)
        return s
    if kind == "varlen":
        total = int(lens.sum())
        s.q = _normal(g, b, hq, hd, dtype=dt)
        s.k, s.v = (_normal(g, total, hkv, hd, dtype=dt) for _ in range(2))
        s.cu_q = torch.arange(b + 1, device=DEVICE, dtype=torch.int32)
        s.cu_k = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(DEVICE, torch.int32)
        s.max_k = int(lens.max())
        return s
    if kind == "dense":
        s.q = _normal(g, b, 1, hq, hd, dtype=dt)
        s.k, s.v = (_normal(g, b, case["hi"], hkv, hd, dtype=dt) for _ in range(2))
        return s
    pool, table = _pages(case, lens, seed)
    s.table = table.to(DEVICE)
    s.seqlens = lens.to(DEVICE, torch.int32)
    cache = _normal(g, 2, pool, case["page_size"], hkv, hd, dtype=dt)
    if case["fp8"]:
        cache = cache.to(torch.float8_e4m3fn)
    if kind == "layer":
        # vLLM's tensors: q, k and v are slices of one fused projection, an
        # fp8 cache is uint8, the output a buffer of the model's.
        qkv = _normal(g, b, (hq + 2 * hkv) * hd, dtype=dt)
        s.q = qkv[:, :hq * hd].view(b, hq, hd)
        s.k = qkv[:, hq * hd:(hq + hkv) * hd].view(b, hkv, hd)
        s.v = qkv[:, (hq + hkv) * hd:].view(b, hkv, hd)
        s.cache = cache.view(torch.uint8) if case["fp8"] else cache
        s.cache_dtype = "fp8" if case["fp8"] else "auto"
        s.k_scale = torch.full((1,), 0.5 if case["fp8"] else 1.0, device=DEVICE)
        s.v_scale = torch.full((1,), 0.25 if case["fp8"] else 1.0, device=DEVICE)
        s.out = torch.empty(b, hq * hd, device=DEVICE, dtype=dt)
        pos = lens - 1
        page = table.gather(1, (pos // case["page_size"])[:, None]).squeeze(1).to(torch.int64)
        s.meta = DecodeMetadata(
            num_actual_tokens=b, max_query_len=1,
            query_start_loc=torch.arange(b + 1, device=DEVICE, dtype=torch.int32),
            max_seq_len=int(lens.max()), seq_lens=s.seqlens, block_table=s.table,
            slot_mapping=(page * case["page_size"] + pos % case["page_size"]).to(DEVICE))
        return s
    s.kc, s.vc = cache[0], cache[1]
    s.q = _normal(g, b, ql, hq, hd, dtype=dt)
    if kind == "verify":
        s.k, s.v = (_normal(g, b, ql, hkv, hd, dtype=dt) for _ in range(2))
        s.accepted = s.seqlens - ql
    if kind == "options":
        s.sinks = torch.randn(hq, generator=g, device=DEVICE) if case["sinks"] else None
        s.alibi = (torch.logspace(-1, -8, hq, base=2.0, device=DEVICE) if case["alibi"]
                   else None)
        s.k_scale = torch.full((1,), 0.5, device=DEVICE) if case["fp8"] else None
        s.v_scale = torch.full((1,), 0.25, device=DEVICE) if case["fp8"] else None
    return s


# ---------------------------------------------------------------------------
# One pass


def run(s):
    if s.kind == "paged":
        return mx.flash_attn_with_kvcache(s.q, s.kc, s.vc, cache_seqlens=s.seqlens,
                                          block_table=s.table)
    if s.kind == "verify":
        # The last step's drafts were rejected: back to the accepted lengths,
        # then the new drafts are appended and verified (which advances them).
        s.seqlens.copy_(s.accepted)
        out = mx.flash_attn_with_kvcache(s.q, s.kc, s.vc, k=s.k, v=s.v, cache_seqlens=s.seqlens,
                                         block_table=s.table, causal=True)
        return {"out": out, "k_cache": s.kc, "v_cache": s.vc, "seqlens": s.seqlens}
    if s.kind == "varlen":
        return mx.flash_attn_varlen_func(s.q, s.k, s.v, s.cu_q, s.cu_k, 1, s.max_k, causal=True)
    if s.kind == "dense":
        return mx.flash_attn_func(s.q, s.k, s.v, causal=True)
    if s.kind == "layer":
        kv_cache_update(s.k, s.v, s.cache, s.meta.slot_mapping, s.cache_dtype, s.k_scale,
                        s.v_scale)
        forward_decode(s.q, s.cache, s.meta, s.out, softmax_scale=s.scale,
                       kv_cache_dtype=s.cache_dtype, k_scale=s.k_scale, v_scale=s.v_scale)
        return {"out": s.out, "cache": s.cache}
    if s.kind == "options":
        c = s.case
        return mx.paged_decode_split(s.q, s.kc, s.vc, s.table, s.seqlens, s.scale,
                                     k_scale=s.k_scale, v_scale=s.v_scale, causal=True,
                                     window_left=c["window"], sinks=s.sinks,
                                     softcap=c["softcap"], alibi_slopes=s.alibi)
    mx.reshape_and_cache(s.key, s.value, s.kc, s.vc, s.slots)
    return {"k_cache": s.kc, "v_cache": s.vc}


def work(case):
    hd, hkv, hq, ql, b = (case[k] for k in ("head_dim", "kv_heads", "q_heads", "q_len", "batch"))
    row = 2 * hkv * hd  # K and V elements of one token
    esz = 1 if case["fp8"] else 2
    if case["kind"] == "write":
        return {"bytes": case["hi"] * (2 * row * 2 + 8), "flops": 0}
    lens = _lengths(case)
    seen = lens if case["window"] < 0 else lens.clamp(max=case["window"] + ql)
    total = int(seen.sum())
    moved = total * row * esz + 2 * b * ql * hq * hd * 2 + 4 * b
    if case["kind"] in ("paged", "verify", "layer", "options"):
        moved += 4 * int(((seen + case["page_size"] - 1) // case["page_size"]).sum())
    if case["kind"] == "verify":  # the drafts' rows are read and written
        moved += 2 * b * ql * row * 2
    elif case["kind"] == "layer":
        moved += b * (row * (2 + esz) + 8)
    return {"bytes": moved, "flops": 4 * total * hq * hd * ql}


def tolerance(case):
    if case["kind"] == "write":
        return "exact"
    # Outputs are rounded once to the 16-bit type and so are the softmax
    # weights; both sides of a comparison carry that rounding.
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits


def _attend(q, k, v, scale, window=-1, softcap=0.0, sinks=None, alibi=None):
    """q [QL, HQ, D] on the last QL of the keys k, v [L, HKV, D], causal; float64."""
    ql, hq, hd = q.shape
    n, hkv = k.shape[0], k.shape[1]
    qh = q.double().reshape(ql, hkv, hq // hkv, hd).permute(1, 2, 0, 3).reshape(hkv, -1, hd)
    kh = k.double().permute(1, 2, 0).contiguous()
    x = torch.matmul(qh.contiguous(), kh).reshape(hq, ql, n) * scale
    if softcap > 0:
        x = softcap * torch.tanh(x / softcap)
    behind = (n - ql + torch.arange(ql, device=q.device)[:, None]
              - torch.arange(n, device=q.device)[None, :])
    if alibi is not None:
        x = x - alibi.double()[:, None, None] * behind.abs()
    hidden = behind < 0
    if window >= 0:
        hidden = hidden | (behind > window)
    x = x.masked_fill(hidden, -math.inf)
    if sinks is not None:
        x = torch.cat([x, sinks.double()[:, None, None].expand(hq, ql, 1)], dim=-1)
    p = torch.softmax(x, dim=-1)[..., :n].reshape(hkv, -1, n)
    o = torch.matmul(p.contiguous(), v.double().permute(1, 0, 2).contiguous())
    return o.reshape(hq, ql, hd).permute(1, 0, 2)


def exact(case, seed):
    s = prepare(case, seed)
    kind, lens = s.kind, s.lens.tolist()
    if kind == "write":
        kc, vc = (torch.zeros_like(c, dtype=torch.float64) for c in (s.kc, s.vc))
        kc.view(-1, *kc.shape[2:])[s.slots] = s.key.double()
        vc.view(-1, *vc.shape[2:])[s.slots] = s.value.double()
        return {"k_cache": kc, "v_cache": vc}
    if kind == "varlen":
        at = s.cu_k.tolist()
        return torch.stack([_attend(s.q[i:i + 1], s.k[at[i]:at[i + 1]], s.v[at[i]:at[i + 1]],
                                    s.scale)[0] for i in range(case["batch"])])
    if kind == "dense":
        return torch.stack([_attend(s.q[i], s.k[i], s.v[i], s.scale)
                            for i in range(case["batch"])])
    ps = case["page_size"]

    def rows(i, n):  # cache rows (flat token index) of sequence i's first n tokens
        pos = torch.arange(n, device=DEVICE)
        return s.table[i].to(torch.int64)[pos // ps] * ps + pos % ps

    if kind == "layer":
        cache = s.cache.view(torch.float8_e4m3fn) if case["fp8"] else s.cache
        kc, vc = (c.reshape(-1, *c.shape[2:]) for c in cache.unbind(0))
        ks, vs = (float(t) if case["fp8"] else 1.0 for t in (s.k_scale, s.v_scale))
        out = []
        for i, n in enumerate(lens):
            at = rows(i, n)
            k, v = kc[at].double(), vc[at].double()
            for side, new, scale in ((k, s.k[i], ks), (v, s.v[i], vs)):
                new = new.float() / scale
                if case["fp8"]:
                    new = new.clamp(-448, 448).to(torch.float8_e4m3fn)
                side[n - 1] = new.double()
            out.append(_attend(s.q[i][None], k * ks, v * vs, s.scale).flatten())
        return {"out": torch.stack(out), "cache": None}
    kc, vc = (c.reshape(-1, *c.shape[2:]) for c in (s.kc, s.vc))
    if kind == "verify":
        for i, n in enumerate(lens):
            at = rows(i, n)[n - case["q_len"]:]
            kc[at], vc[at] = s.k[i], s.v[i]
    more = {}
    ks = vs = 1.0
    if kind == "options":
        more = dict(window=case["window"], softcap=case["softcap"], sinks=s.sinks, alibi=s.alibi)
        ks, vs = (float(t) if case["fp8"] else 1.0 for t in (s.k_scale, s.v_scale))
    out = []
    for i, n in enumerate(lens):
        at = rows(i, n)
        out.append(_attend(s.q[i], kc[at].double() * ks, vc[at].double() * vs, s.scale, **more))
    out = torch.stack(out)
    if kind != "verify":
        return out
    return {"out": out, "k_cache": kc.reshape(s.kc.shape).double(),
            "v_cache": vc.reshape(s.vc.shape).double(), "seqlens": None}
