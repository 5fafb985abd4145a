"""Ragged batches through the batched decode (cf_kv_paged_attention_batched_async): with splits = 0 a batch of several
sequences runs as a span launch, which lays the chain pairs of all sequences end to end over one workgroup per CU. Every
row is compared with the split launch of the same descriptor (splits = 1, which takes each sequence by itself) and the
rows of some sequences with a float64 softmax over the INT8-quantised pages in torch.

Shapes sit where the spans can go wrong: sequences without visible tokens (first, last, in a row), fewer pairs than
workgroups and than wavefronts, sequences far longer than a workgroup's share, ends on and off the pair boundary, one KV
head and many, head_dim 64, both codecs, raw INT8 groups inside a rANS pool, a query in the middle of its context."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RAGGED = [1, 64, 65, 128, 129, 3100, 16, 700, 191, 192, 193, 257] + [1, 30, 64, 900, 5, 128, 1000, 2]
MANY = [7, 64, 100, 65] * 34 + [3100, 1, 129, 64]


def _reference(q, k, v, tokens, scale):
    """float64 attention of q [H, g, D] over the quantised pages of k, v [H, T, D]."""
    import torch
    H, T, D = k.shape
    pad = (-T) % 16

    def deq(x):
        x = torch.from_numpy(np.pad(x, ((0, 0), (0, pad), (0, 0)))).view(H, -1, 16, D)
        m = x.abs().amax(dim=(2, 3), keepdim=True)
        s = torch.where(m == 0, torch.ones_like(m), m / 127.0)
        return (torch.round(x / s).double() * s.double()).view(H, -1, D)[:, :tokens]

    w = torch.softmax(torch.matmul(torch.from_numpy(q).double(), deq(k).transpose(1, 2)) * scale, -1)
    return torch.matmul(w, deq(v)).numpy()


@pytest.mark.parametrize("codec,H,gqa,D,lens,raw", [
    ("rans", 8, 4, 128, RAGGED, None),                      # one long sequence over many workgroups
    ("rans", 1, 1, 64, MANY, None),                         # one KV head: every CU's workgroup on it
    ("rans", 7, 3, 64, RAGGED[::-1], None),
    ("rans", 16, 2, 64, [1024] * 25, None),                 # all alike, no divisor of anything
    ("rans", 8, 4, 128, ([1100, 3, 70] * 17)[:50], None),   # more units than CUs
    ("rans", 8, 4, 128, RAGGED, {0: 1, 1: 1, 5: 9, 7: 3, 15: 15}),  # raw groups, odd counts and whole sequences
    ("int8", 8, 2, 64, RAGGED, None),
    ("int8", 8, 4, 128, RAGGED[::-1], None),
])
@pytest.mark.parametrize("hide", [(), (0, 1), (-1,)])
def test_spans_match_the_split_launch(codec, H, gqa, D, lens, raw, hide):
    import torch
    from chromofold_amd import kv
    print(f"case {codec} H={H} gqa={gqa} D={D} lens={lens} raw={raw} hide={hide}", flush=True)
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(D + H + len(lens))
    S = len(lens)
    data = [tuple(rng.standard_normal((H, T, D)).astype(np.float32) for _ in range(2)) for T in lens]
    big = max(range(S), key=lambda s: lens[s])
    tables = None
    cdc = kv.CODEC_INT8
    if codec == "rans":
        cdc = kv.CODEC_RANS_HYBRID
        n = lens[big] // 16 * 16
        tables = np.concatenate([kv.build_table(x[h][:min(n, 256)].reshape(-1, 16, D)) for h in range(H) for x in data[big]])
    kvb = kv.build_batched(cdc, lambda s: data[s], S, H, np.array(lens), D, tables, dev,
                           encoder="host" if raw else "device", raw_groups=raw)
    q = rng.standard_normal((S, H * gqa, D)).astype(np.float32)
    pos = np.array(lens, np.int64) - 1
    pos[S // 2] //= 2  # a query inside its context
    tok = np.array(lens, np.int64)
    for s in hide:
        tok[s] = 0  # nothing visible
    kvb.seq_tokens = torch.from_numpy(tok.astype(np.int32)).to(dev)
    qd, pd = torch.from_numpy(q).to(dev), torch.from_numpy(pos.astype(np.int32)).to(dev)
    scale = 1.0 / np.sqrt(D)
    assert kvb.desc(qd, qd, pd, scale).workspace_bytes > 0, "one split and no span launch"
    outs = []
    for splits in (0, 1):
        out = torch.full(q.shape, float("nan"), device=dev)
        kvb.workspace = None
        kvb.attention(qd, out, pd, scale, splits=splits)
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    assert np.isfinite(outs[0]).all()
    norm = np.maximum(np.linalg.norm(outs[1], axis=-1), 1e-6)
    # the same sums grouped otherwise: fp32 rounding of the running softmax and the f16 hi + lo weights (5e-6 of a row
    # at 32k tokens)
    err = np.linalg.norm(outs[0] - outs[1], axis=-1) / norm
    assert err.max() <= 1e-5, (int(err.max(axis=1).argmax()), float(err.max()))
    for s in hide:
        assert not outs[0][s].any()
    for s in {0, S // 2, S - 1, big}:
        n = int(min(tok[s], pos[s] + 1))
        if n == 0:
            continue
        ref = _reference(q[s].reshape(H, gqa, D), *data[s], n, scale).reshape(H * gqa, D)
        err = np.linalg.norm(outs[0][s] - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
        assert err.max() <= 2e-5, (s, float(err.max()))


def test_span_in_a_graph_and_with_a_small_workspace():
    """Replays of a captured span launch (with eager launches of other lengths between them, over the same workspace)
    equal the eager result bit for bit; a workspace too small for the span states runs the split launch instead."""
    import torch
    from chromofold_amd import kv
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(5)
    H, gqa, D, lens = 8, 4, 128, RAGGED
    data = [tuple(rng.standard_normal((H, T, D)).astype(np.float32) for _ in range(2)) for T in lens]
    tables = np.concatenate([kv.build_table(x[h][:64].reshape(-1, 16, D)) for h in range(H) for x in data[5]])
    kvb = kv.build_batched(kv.CODEC_RANS_HYBRID, lambda s: data[s], len(lens), H, np.array(lens), D, tables, dev,
                           encoder="device")
    q = torch.from_numpy(rng.standard_normal((len(lens), H * gqa, D)).astype(np.float32)).to(dev)
    out = torch.empty_like(q)
    pos = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
    scale = 1.0 / np.sqrt(D)
    desc = kvb.desc(q, out, pos, scale)
    run = lambda: kvb.attention(q, out, pos, scale, desc=desc)  # noqa: E731
    run()
    torch.cuda.synchronize()
    eager = out.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run()
    full = kvb.seq_tokens.clone()
    for i in range(4):
        kvb.seq_tokens.copy_(torch.minimum(full, torch.arange(len(lens), device=dev) * (40 + i)))
        run()
        kvb.seq_tokens.copy_(full)
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), i
    desc.workspace_bytes = int(len(lens) * H * 12 * 4 * (D + 2) * 4)  # room for split partials, not for spans
    out.fill_(float("nan"))
    assert desc.workspace_bytes < kvb.workspace.numel()
    run()
    torch.cuda.synchronize()
    assert float((out - eager).norm() / eager.norm()) <= 1e-5


def test_calls_on_two_streams_have_a_workspace_each():
    """Overlapping calls of one batch on two streams, over shapes that run as spans, give the results of calls in turn."""
    import torch
    from chromofold_amd import kv
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(6)
    H, gqa, D, lens = 4, 2, 64, [3000, 200, 900, 64] * 10
    data = [tuple(rng.standard_normal((H, T, D)).astype(np.float32) for _ in range(2)) for T in lens]
    kvb = kv.build_batched(kv.CODEC_INT8, lambda s: data[s], len(lens), H, np.array(lens), D, None, dev, encoder="device")
    pos = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
    qs = [torch.from_numpy(rng.standard_normal((len(lens), H * gqa, D)).astype(np.float32)).to(dev) for _ in range(2)]
    want = [torch.empty_like(q) for q in qs]
    for q, o in zip(qs, want):
        kvb.attention(q, o, pos, 0.125)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    ptrs = [kvb.desc(qs[0], want[0], pos, 0.125, stream=s).workspace for s in streams]
    assert ptrs[0] != ptrs[1] and ptrs[0] == kvb.desc(qs[0], want[0], pos, 0.125, stream=streams[0]).workspace
    got = [torch.empty_like(q) for q in qs]
    torch.cuda.synchronize()
    for _ in range(20):
        for s, q, o in zip(streams, qs, got):
            kvb.attention(q, o, pos, 0.125, stream=s)
    torch.cuda.synchronize()
    for o, w in zip(got, want):
        assert torch.equal(o, w)
