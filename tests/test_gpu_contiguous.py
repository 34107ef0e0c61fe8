"""Keys in consecutive rows read in place (dense caches and packed sequences):
the operator's contiguous_decode against the reference port, and the paged
route of the same call, over the layouts both take."""

from __future__ import annotations

import pytest
import torch

import mxflashattn_amd as mx
from mxflashattn_amd import native
from oracle import reference_port

TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}

pytestmark = pytest.mark.gpu


def randn(*shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def close(got, expected, dtype):
    err = (got.float().cpu() - expected.float()).abs().max().item()
    assert err <= TOL[dtype], err


def both_routes(monkeypatch, taken, call):
    """The call as consecutive rows (the operator takes it) and through the paged route."""
    taken.clear()
    out = call()
    assert taken[-1] == "contiguous_decode"
    assert mx.get_last_dispatch_info().backend == mx.BACKEND_MI355X
    with monkeypatch.context() as m:
        m.setattr(native, "USE_TORCH_OP", False)
        return out, call()


@pytest.mark.parametrize("hd,gq,dtype", [(64, 1, torch.float16), (64, 8, torch.bfloat16),
                                         (128, 2, torch.float16), (128, 4, torch.bfloat16),
                                         (128, 16, torch.bfloat16)])
@pytest.mark.parametrize("wide", [False, True], ids=["int32", "int64"])
def test_packed_rows(device, monkeypatch, taken, hd, gq, dtype, wide):
    hkv = 3
    lens = [1, 15, 16, 17, 700, 33, 1900, 5]
    rows = [1, 1, 0, 1, 1, 0, 1, 1]  # sequences 2 and 5 have no query row
    kv = randn(sum(lens), 2, hkv, hd, dtype=dtype, seed=hd + gq)  # K and V rows interleaved
    q = randn(sum(rows), hkv * gq + 1, hd, dtype=dtype, seed=gq)[:, 1:]
    cu_q = torch.tensor([0, *torch.tensor(rows).cumsum(0).tolist()])
    cu_k = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()])
    ref = reference_port.attention_varlen(q.float(), kv[:, 0].float(), kv[:, 1].float(),
                                          cu_q.tolist(), cu_k.tolist(), softmax_scale=hd ** -0.5)
    dt = torch.int64 if wide else torch.int32
    d = kv.to(device)
    qd = torch.empty(sum(rows), hkv * gq + 1, hd, dtype=dtype, device=device)
    qd[:, 1:] = q.to(device)
    out, paged = both_routes(monkeypatch, taken, lambda: mx.flash_attn_varlen_func(
        qd[:, 1:], d[:, 0], d[:, 1], cu_q.to(device, dt), cu_k.to(device, dt), 1, max(lens)))
    close(out, ref, dtype)
    assert torch.equal(out, paged)  # the same tiles, ranges and arithmetic


@pytest.mark.parametrize("hd,dtype", [(64, torch.float16), (64, torch.bfloat16),
                                      (128, torch.bfloat16)])
@pytest.mark.parametrize("gq", [1, 4, 8, 16])
@pytest.mark.parametrize("form", ["packed", "dense"])
def test_short_sequences_round_no_more_than_their_pages(device, monkeypatch, taken, hd, dtype, gq,
                                                        form):
    """Short enough for the per-sequence kernel, which pages of less than a tile
    never took: a wave of it walks several tiles, where their split has about one
    a piece. Against 64 bits the error is the rounding of P, sampled over 49,000
    outputs and more (0.3 % of noise), held to 2 %; with one reference maximum
    for a wave's tiles it was 8-17 % larger."""
    lens = [97, 130, 207, 301] if form == "packed" else [301] * 4
    err = {"rows": 0.0, "pages": 0.0}
    for seed in range(max(1, 96 // gq)):
        k, v = (randn(sum(lens), 2, hd, dtype=dtype, seed=2 * seed + i).to(device) for i in (0, 1))
        q = randn(4, 2 * gq, hd, dtype=dtype, seed=1000 + seed).to(device)
        if form == "packed":
            cu_q, cu_k = (torch.tensor([0, *torch.tensor(x).cumsum(0).tolist()], device=device)
                          for x in ([1] * 4, lens))
            got = both_routes(monkeypatch, taken, lambda: mx.flash_attn_varlen_func(
                q, k, v, cu_q, cu_k, 1, max(lens)))
        else:
            got = both_routes(monkeypatch, taken, lambda: mx.flash_attn_func(
                q[:, None], k.unflatten(0, (4, -1)), v.unflatten(0, (4, -1)), causal=True))
        want, at = [], 0
        for b, n in enumerate(lens):
            ki, vi = (t[at:at + n].double().permute(1, 0, 2) for t in (k, v))
            s = torch.matmul(q[b].double().view(2, gq, hd), ki.transpose(1, 2).contiguous())
            want.append(torch.matmul(torch.softmax(s * hd ** -0.5, -1), vi.contiguous()))
            at += n
        want = torch.stack(want).view(4, 2 * gq, hd)
        for name, out in zip(err, got):
            err[name] += (out.view_as(q).double() - want).square().sum().item()
    assert err["rows"] <= 1.02 ** 2 * err["pages"], err


@pytest.mark.parametrize("seq", [1, 15, 47, 96, 1025, 2048])
@pytest.mark.parametrize("hd,gq,ql,dtype", [(64, 2, 1, torch.float16), (128, 4, 1, torch.bfloat16),
                                            (128, 1, 3, torch.bfloat16), (64, 4, 9, torch.float16),
                                            (128, 4, 16, torch.bfloat16)])
def test_dense_rows(device, monkeypatch, taken, seq, hd, gq, ql, dtype):
    if ql > seq:
        pytest.skip("fewer keys than query tokens")
    kv = randn(3, seq, 2, 2, hd, dtype=dtype, seed=seq)  # token rows of K and V interleaved
    q = randn(3, ql, 2 * gq, hd, dtype=dtype, seed=ql)
    ref = reference_port.attention_batched(q.float(), kv[:, :, 0].float(), kv[:, :, 1].float(),
                                           softmax_scale=hd ** -0.5, causal=True)
    d = kv.to(device)
    out, paged = both_routes(monkeypatch, taken, lambda: mx.flash_attn_func(
        q.to(device), d[:, :, 0], d[:, :, 1], causal=True))
    close(out, ref, dtype)
    close(paged, ref, dtype)
    if ql * gq <= 16:  # one launch: the pages' tiles, ranges and arithmetic
        assert torch.equal(out, paged)
    # The cache entry point: lengths of its own, some empty, into a given output.
    lens = torch.tensor([seq, (seq + 1) // 2, 0], dtype=torch.int32)
    buf = torch.full((3, ql, 2 * gq + 3, hd), 7.0, device=device, dtype=dtype)
    got = mx.flash_attn_with_kvcache(q.to(device), d[:, :, 0], d[:, :, 1],
                                     cache_seqlens=lens.to(device), causal=True,
                                     out=buf[:, :, 1:-2])
    assert taken[-1] == "contiguous_decode"
    assert got.data_ptr() == buf[:, :, 1:-2].data_ptr()
    for b in range(3):
        n = int(lens[b])
        want = torch.zeros(ql, 2 * gq, hd) if n == 0 else reference_port.attention_single(
            q[b].float(), kv[b, :n, 0].float(), kv[b, :n, 1].float(), softmax_scale=hd ** -0.5,
            causal=True)
        close(got[b], want, dtype)
    assert (buf[:, :, :1] == 7).all() and (buf[:, :, -2:] == 7).all()


def test_offsets_that_name_no_keys_read_nothing_outside(device):
    # The operator itself, past the API's checks: offsets that run backwards,
    # start before the keys or end after them are held to the rows that exist.
    op = native.torch_op()
    k, v = (randn(100, 2, 64, dtype=torch.float16, seed=s).to(device) for s in (5, 6))
    q = randn(4, 4, 64, dtype=torch.float16, seed=7).to(device)
    cu_q = torch.arange(5, dtype=torch.int32, device=device)
    cu_k = torch.tensor([-50, 90, 5000, 40, 100], dtype=torch.int32, device=device)
    out = op.contiguous_decode(q, k, v, 0.125, False, 128, cu_q, cu_k)
    ref = [(0, 90), (90, 100), (0, 0), (40, 100)]
    for b, (a, e) in enumerate(ref):
        want = torch.zeros(4, 64) if a == e else reference_port.attention_single(
            q[b:b + 1].float().cpu(), k[a:e].float().cpu(), v[a:e].float().cpu(),
            softmax_scale=0.125)[0]
        close(out[b], want, torch.float16)


def test_a_row_that_several_sequences_name_takes_one_of_them(device):
    # Offsets the API refuses once it has read them; the kernels are out by then.
    # 200 sequences, every other one of query row 0: the first of all keys, the
    # last (in another wave) of the last key. A first row of one with the length
    # of the other would pass the keys' end.
    op = native.torch_op()
    k, v = (randn(100, 2, 64, dtype=torch.float16, seed=s).to(device) for s in (5, 6))
    q = randn(1, 4, 64, dtype=torch.float16, seed=7).to(device)
    cu_q = torch.arange(201, dtype=torch.int32, device=device) % 2
    cu_k = torch.tensor([0, 100] + [50, 60] * 98 + [99, 100, 100], dtype=torch.int32,
                        device=device)
    out = op.contiguous_decode(q, k, v, 0.125, False, 100, cu_q, cu_k)
    want = [reference_port.attention_single(q.float().cpu(), k[a:e].float().cpu(),
                                            v[a:e].float().cpu(), softmax_scale=0.125)
            for a, e in ((0, 100), (50, 60), (99, 100))]
    errs = [(out.float().cpu() - w).abs().max().item() for w in want]
    assert min(errs) <= TOL[torch.float16], errs
    with pytest.raises(ValueError, match="cu_seqlens_q must start at zero"):
        mx.flash_attn_varlen_func(q, k, v, cu_q, cu_k, 1, 100)


def test_packed_offsets_are_checked_after_the_launch(device, taken):
    """Offsets the API rejects raise the same errors as before the kernels
    went out first, leave the next call right, and name no row outside."""
    k, v = (randn(60, 2, 64, dtype=torch.float16, seed=s).to(device) for s in (8, 9))
    q = randn(3, 4, 64, dtype=torch.float16, seed=10).to(device)
    good = torch.tensor([0, 20, 21, 60])

    def call(cu_q, cu_k, max_q=1, max_k=60):
        return mx.flash_attn_varlen_func(q, k, v, torch.tensor(cu_q).to(device),
                                         torch.as_tensor(cu_k).to(device), max_q, max_k)

    for cu_q, cu_k, match in (([0, 1, 2, 3], [0, 20, 70, 60], "cu_seqlens_k must be monotonically"),
                              ([0, 1, 2, 3], [0, 20, 20, 60], "must be non-empty"),
                              ([0, 1, 2, 3], [0, 20, 21, 59], "cu_seqlens_k must start at zero"),
                              ([0, 2, 2, 3], good, "cu_seqlens_q contains a sequence longer"),
                              ([1, 1, 2, 3], good, "cu_seqlens_q must start at zero"),
                              ([0, 1, 2, 3, 3], good, "same batch size")):
        taken.clear()
        with pytest.raises(ValueError, match=match):
            call(cu_q, cu_k)
        # The last one's vectors differ in length: nothing goes out early.
        assert taken[-1:] == (["contiguous_decode"] if len(cu_q) == 4 else ["PackedOffsets"])
    with pytest.raises(ValueError, match="cu_seqlens_k contains a sequence longer"):
        call([0, 1, 2, 3], good, max_k=38)
    taken.clear()
    out = call([0, 1, 2, 3], good)
    assert taken == ["PackedOffsets", "contiguous_decode"]
    ref = reference_port.attention_varlen(q.float().cpu(), k.float().cpu(), v.float().cpu(),
                                          [0, 1, 2, 3], good.tolist(), softmax_scale=0.125)
    close(out, ref, torch.float16)


def test_packed_offsets_reach_the_host(device):
    op = native.torch_op()
    k, v = (randn(500, 1, 64, dtype=torch.bfloat16, seed=s).to(device) for s in (1, 2))
    for n, dt in ((3, torch.int32), (250, torch.int64), (3, torch.int64)):
        q = randn(n, 2, 64, dtype=torch.bfloat16, seed=n).to(device)
        cu_q = torch.arange(n + 1)
        cu_k = torch.linspace(0, 500, n + 1).long()
        offsets = op.PackedOffsets()
        assert offsets.get() is None
        out = op.contiguous_decode(q, k, v, 0.125, False, 500, cu_q.to(device, dt),
                                   cu_k.to(device, dt), offsets=offsets)
        assert out is not None
        assert offsets.get() == (cu_q.tolist(), cu_k.tolist())


# One lane's, four lanes' and the LDS tile scan; past one pass of the rows launch.
@pytest.mark.parametrize("seqs", [65, 257, 1100])
@pytest.mark.parametrize("hd,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("longest", [59, 801])  # the per-sequence kernel, the split kernel
def test_many_sequences(device, monkeypatch, taken, seqs, hd, dtype, longest):
    g = torch.Generator().manual_seed(seqs)
    lens = torch.randint(1, 60, (seqs,), generator=g)
    rows = torch.randint(0, 4, (seqs,), generator=g).clamp(max=1)  # a quarter without a row
    lens[seqs // 2], rows[seqs // 2] = longest, 1
    k, v = (randn(int(lens.sum()), 2, hd, dtype=dtype, seed=s) for s in (1, 2))
    q = randn(int(rows.sum()), 4, hd, dtype=dtype, seed=3)
    cu_q, cu_k = (torch.nn.functional.pad(t.cumsum(0), (1, 0)) for t in (rows, lens))
    ref = reference_port.attention_varlen(q.float(), k.float(), v.float(), cu_q.tolist(),
                                          cu_k.tolist(), softmax_scale=hd ** -0.5)
    out, paged = both_routes(monkeypatch, taken, lambda: mx.flash_attn_varlen_func(
        q.to(device), k.to(device), v.to(device), cu_q.to(device), cu_k.to(device), 1,
        int(lens.max())))
    close(out, ref, dtype)
    if longest == 801:
        assert torch.equal(out, paged)
    g = torch.Generator(device=device).manual_seed(seqs)
    kd, vd = (torch.randn(seqs, longest, 1, hd, generator=g, device=device).to(dtype)
              for _ in range(2))
    qd = torch.randn(seqs, 1, 4, hd, generator=g, device=device).to(dtype)
    some = torch.arange(0, seqs, 37, device=device)
    ref = reference_port.attention_batched(*(t[some].float().cpu() for t in (qd, kd, vd)),
                                           softmax_scale=hd ** -0.5, causal=True)
    out, paged = both_routes(monkeypatch, taken, lambda: mx.flash_attn_func(qd, kd, vd,
                                                                           causal=True))
    close(out[some], ref, dtype)
    close(out, paged.cpu(), dtype)
    if longest == 801:
        assert torch.equal(out, paged)


def test_a_sequence_past_4_gib(device, monkeypatch, taken):
    # Token rows 128 KiB apart: the last ones lie past 2^32 bytes from the first.
    seq, hd = 34001, 64
    buf = torch.empty(seq, 65536, dtype=torch.bfloat16, device=device)
    kv = randn(seq, 2 * hd, dtype=torch.bfloat16, seed=1)
    buf[:, :2 * hd] = kv.to(device)
    k, v = (buf[:, i * hd:(i + 1) * hd].unsqueeze(1) for i in (0, 1))
    q = randn(1, 4, hd, dtype=torch.bfloat16, seed=2)
    # The last keys outweigh the others, so the output is mostly theirs.
    q[0, :2] = kv[-1, :hd]
    ref = reference_port.attention_single(q.float(), kv[:, None, :hd].float(),
                                          kv[:, None, hd:].float(), softmax_scale=hd ** -0.5)
    out, paged = both_routes(monkeypatch, taken, lambda: mx.flash_attn_func(
        q.to(device)[None], k[None], v[None], causal=True))
    close(out[0], ref, torch.bfloat16)
    assert torch.equal(out, paged)
    cu = torch.tensor([0, 100, seq], device=device)
    got = mx.flash_attn_varlen_func(q.to(device).expand(2, 4, hd).contiguous(), k, v,
                                    torch.arange(3, device=device), cu, 1, seq)
    want = reference_port.attention_single(q.float(), kv[100:, None, :hd].float(),
                                           kv[100:, None, hd:].float(), softmax_scale=hd ** -0.5)
    close(got[1:], want, torch.bfloat16)


@pytest.mark.parametrize("ql,seq", [(1, 3001), (16, 3001), (1, 96)])
def test_dense_keys_from_a_graph(device, taken, ql, seq):
    # First rows and lengths are memory of the graph; other calls in between,
    # on the capture's stream and off it, do not change a replay.
    k, v = (randn(4, seq, 2, 128, dtype=torch.bfloat16, seed=s).to(device) for s in (1, 2))
    q = randn(4, ql, 8, 128, dtype=torch.bfloat16, seed=3).to(device)
    stream = torch.cuda.Stream(device)
    with torch.cuda.stream(stream):
        want = mx.flash_attn_func(q, k, v, causal=True)
    torch.cuda.synchronize()
    taken.clear()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = mx.flash_attn_func(q, k, v, causal=True)
    assert taken == ["contiguous_decode"]
    cu = torch.tensor([0, 20, seq], device=device)
    for _ in range(3):
        out.fill_(7)
        for s in (stream, torch.cuda.current_stream()):
            with torch.cuda.stream(s):
                mx.flash_attn_varlen_func(q[0, 0].expand(2, 8, 128).contiguous(), k[0], v[0],
                                          torch.arange(3, device=device), cu, 1, seq)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_calls_on_several_streams_and_threads(device):
    """First rows and lengths are a stream's own: calls of different sizes in
    flight on four streams, one thread each, give what they give alone."""
    from concurrent.futures import ThreadPoolExecutor

    def inputs(i):
        lens = torch.arange(1 + 3 * i, 41 + 3 * i) * (1 + i) % 300 + 1
        cu_k = torch.nn.functional.pad(lens.cumsum(0), (1, 0))
        k, v = (randn(int(lens.sum()), 2, 64, dtype=torch.float16, seed=10 * i + s).to(device)
                for s in (0, 1))
        q = randn(40, 4, 64, dtype=torch.float16, seed=10 * i + 2).to(device)
        return q, k, v, torch.arange(41, device=device), cu_k.to(device), 1, int(lens.max())

    cases = [inputs(i) for i in range(4)]
    want = [mx.flash_attn_varlen_func(*c) for c in cases]
    streams = [torch.cuda.Stream(device) for _ in cases]
    torch.cuda.synchronize()

    def run(i):
        with torch.cuda.stream(streams[i]):
            dense = (cases[i][0][None, :1], cases[i][1][None, :77], cases[i][2][None, :77])
            return [(mx.flash_attn_varlen_func(*cases[i]), mx.flash_attn_func(*dense, causal=True))
                    for _ in range(25)]

    with ThreadPoolExecutor(4) as pool:
        got = list(pool.map(run, range(4)))
    torch.cuda.synchronize()
    for i, outs in enumerate(got):
        assert all(torch.equal(packed, want[i]) for packed, _ in outs)
        assert all(torch.equal(dense, outs[0][1]) for _, dense in outs)
