"""Performance cases of the library: the calls a serving or search program makes, over the sizes it makes them at.

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges, `prepare` builds what the program already
holds (sealed pages, coded weights, an index, the step's inputs), `run` is one pass through the public entry points,
`work` the bytes and operations the pass cannot do without, `exact` the 64-bit answer in plain torch.

Kinds of case and what each stands for:
  decode    one token per sequence over entropy-coded (or INT8) paged K/V: a serving step of one layer. Llama-3-8B's
            layer shape (8 KV heads, 32 query heads, head_dim 128) unless the case says otherwise; contexts are ragged
            as in any real batch, except where a long-context batch is padded to one length.
  cascade   the same step when every sequence starts with one long shared prompt (stored once, as INT8 groups).
  seal      sealing freshly computed K/V on the device: a prefill's pages, or the groups a decode step completed.
  matmul    y = x W^T over pair-rANS int4 weights: one token (decode) up to a batch of tokens.
  nibble    the multi-sequence resolver: one batch of decode items and short prefill chunks over int4 pages.
  seam      the llama adapter: a chunk of 64 prompt tokens over fixed-width int4/int8 pages and a dense tail.
  search    FM-index: the range of each pattern and the text position of its first row.
  wavelet   RRR wavelet matrix (4-ary layout): access and rank queries.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from chromofold_amd import _abi as A
from chromofold_amd import kv, llama, qw, search, sealkv

DEV = "cuda:0"


def listed():
    return [
        # one interactive chat: one sequence at ~2k tokens, where latency counts
        {"name": "decode_one", "kind": "decode", "codec": "rans", "seqs": 1, "lo": 2003, "hi": 2003, "kvh": 8, "gqa": 4,
         "hd": 128, "lens": 1},
        # an ordinary serving batch: 48 sequences of 150 to 8000 tokens
        {"name": "decode_ragged", "kind": "decode", "codec": "rans", "seqs": 48, "lo": 150, "hi": 8000, "kvh": 8,
         "gqa": 4, "hd": 128, "lens": 2},
        # a small model (head_dim 64, 2 query heads per KV head) served with the decode-free INT8 codec
        {"name": "decode_hd64_int8", "kind": "decode", "codec": "int8", "seqs": 40, "lo": 200, "hi": 6000, "kvh": 4,
         "gqa": 2, "hd": 64, "lens": 3},
        # the long-context batch: 32 sequences at 32k tokens
        {"name": "decode_32x32k", "kind": "decode", "codec": "rans", "seqs": 32, "lo": 32768, "hi": 32768, "kvh": 8,
         "gqa": 4, "hd": 128, "lens": 4},
        # 256 users of one application: an 8192-token system prompt and 512 tokens of their own
        {"name": "cascade_256", "kind": "cascade", "seqs": 256, "shared": 8192, "lo": 512, "hi": 512, "kvh": 8, "gqa": 4,
         "hd": 128, "lens": 5},
        # sealing what a prefill of 16 prompts left behind (ragged last groups)
        {"name": "seal_prefill", "kind": "seal", "codec": "rans", "seqs": 16, "lo": 700, "hi": 4096, "kvh": 8, "hd": 128,
         "lens": 6},
        # a projection of a 4096-wide model for one decoded token
        {"name": "matmul_b1", "kind": "matmul", "rows": 4096, "cols": 4096, "batch": 1},
        # the wide down-projection for a batch of 48 tokens
        {"name": "matmul_wide_b48", "kind": "matmul", "rows": 4096, "cols": 14336, "batch": 48},
        # continuous batching over int4 pages: 24 decode items and 2 prefill chunks of 16 tokens
        {"name": "nibble_batch", "kind": "nibble", "seqs": 26, "lo": 500, "hi": 12000, "kvh": 8, "gqa": 4, "hd": 128,
         "chunks": 2, "chunk": 16, "dtype": "bf16", "lens": 7},
        # llama.cpp's prompt processing: 64 query tokens, 2 KV / 14 query heads, int4 pages of 32 tokens
        {"name": "seam_prefill", "kind": "seam", "tokens": 6000, "kvh": 2, "gqa": 7, "hd": 64, "queries": 64, "bits": 4,
         "page": 32},
        # phrase search in a 16.8M-token corpus: 400k patterns of 4 to 24 tokens
        {"name": "search_16m", "kind": "search", "n": (1 << 24) - 1, "patterns": 400000, "lmin": 4, "lmax": 24},
        # token statistics of a 1M-token stream: 1M access and 1M rank queries
        {"name": "wavelet_1m", "kind": "wavelet", "n": 1 << 20, "queries": 1 << 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "cascade", "seal", "matmul", "matmul", "nibble", "seam", "search",
                       "wavelet"])
    lens = rng.randrange(1 << 30)
    if kind == "decode":
        while True:
            seqs, hi = _log(rng, 1, 96), _log(rng, 64, 32768)
            c = {"kind": kind, "codec": rng.choice(["rans", "rans", "int8"]), "seqs": seqs,
                 "lo": hi if rng.random() < 0.25 else max(1, int(hi * rng.uniform(0.02, 0.9))), "hi": hi,
                 "kvh": rng.choice([2, 4, 8]), "gqa": rng.choice([1, 2, 3, 4, 4]), "hd": rng.choice([64, 128, 128]),
                 "lens": lens}
            if sum(_lens(c)) * c["kvh"] * c["hd"] <= 32 * 32768 * 8 * 128:
                return c
    if kind == "cascade":
        hi = _log(rng, 64, 1024)
        return {"kind": kind, "seqs": _log(rng, 5, 256), "shared": 64 * _log(rng, 4, 128),
                "lo": rng.randint(1, hi), "hi": hi, "kvh": rng.choice([2, 4, 8]), "gqa": rng.choice([2, 3, 4]),
                "hd": 128, "lens": lens}
    if kind == "seal":
        hi = _log(rng, 32, 4096)
        return {"kind": kind, "codec": rng.choice(["rans", "rans", "int8"]), "seqs": _log(rng, 1, 32),
                "lo": rng.randint(1, hi), "hi": hi, "kvh": rng.choice([2, 4, 8]), "hd": rng.choice([64, 128, 128]),
                "lens": lens}
    if kind == "matmul":
        while True:
            rows, cols = _log(rng, 1000, 16000), _log(rng, 1000, 16000)
            if rng.random() < 0.7:
                rows, cols = max(512, rows // 256 * 256), max(512, cols // 256 * 256)
            if rows * cols <= 4096 * 14336:
                return {"kind": kind, "rows": rows, "cols": cols, "batch": _log(rng, 1, 64)}
    if kind == "nibble":
        hi, seqs = _log(rng, 64, 12000), _log(rng, 1, 40)
        return {"kind": kind, "seqs": seqs, "lo": rng.randint(20, hi), "hi": hi, "kvh": rng.choice([2, 4, 8]),
                "gqa": rng.choice([1, 2, 4]), "hd": rng.choice([64, 128, 128]), "chunks": min(seqs, rng.randrange(3)),
                "chunk": rng.choice([8, 16]), "dtype": rng.choice(["bf16", "f32"]), "lens": lens}
    if kind == "seam":
        return {"kind": kind, "tokens": _log(rng, 100, 16000), "kvh": 2, "gqa": rng.choice([4, 7]),
                "hd": rng.choice([64, 128]), "queries": rng.choice([1, 8, 64]), "bits": rng.choice([4, 4, 8]), "page": 32}
    if kind == "search":
        lmin = rng.randint(1, 8)
        return {"kind": kind, "n": _log(rng, 1 << 16, 1 << 24) - 1, "patterns": _log(rng, 200, 400000), "lmin": lmin,
                "lmax": lmin + rng.randint(0, 24)}
    return {"kind": kind, "n": _log(rng, 1 << 13, 1 << 21), "queries": _log(rng, 1 << 8, 1 << 20)}


def _scale(m, top):
    """max / top (1 for an all-zero block), by an IEEE division: torch turns a division by a plain number on the GPU
    into a product with its reciprocal."""
    return torch.where(m == 0, torch.ones_like(m), m / torch.full_like(m, top))


def _lens(case):
    """The context lengths of a batch: log-uniform in [lo, hi], a property of the case (not of the seed)."""
    r = random.Random(case["lens"])
    return [_log(r, case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(0xC0DE + 7919 * seed + 104729 * salt)
    return g


# ---------------------------------------------------------------------------------- coded paged K/V (decode, cascade, seal)
def _pages_of(lens):
    return [(t + 15) // 16 for t in lens]


def _kv_values(seed, npages, hd, salt=0):
    """Page-major K and V [npages, 16, hd] fp32: keys with a spread of channel magnitudes, as after a rotary
    projection, values N(0, 1)."""
    g = _gen(seed, salt)
    ch = torch.exp(0.25 * torch.randn(hd, generator=g, device=DEV))
    k = torch.randn((npages, 16, hd), generator=g, device=DEV)
    k *= ch
    return k, torch.randn((npages, 16, hd), generator=g, device=DEV)


def _groups(lens, kvh, skip=None, base=0):
    """Group lists of a batch whose pages are stored sequence by sequence, head by head: first page, page count, head,
    continues flag, per-page token counts, and each sequence's slice of the group list. `skip` = groups of every
    sequence that lie in a shared prefix (their indices precede the sequence's own)."""
    first, counts, heads, cont, tc, at, page = [], [], [], [], [], [], base
    n = 0
    for t in lens:
        npg = (t + 15) // 16
        ngr = (npg + 3) // 4
        gi = np.arange(ngr)
        fl = kv.pair_flags(gi + (skip or 0), skip or 0)
        tcs = np.full(npg, 16, np.int32)
        tcs[-1] = t - 16 * (npg - 1)
        for h in range(kvh):
            first.append(page + 4 * gi)
            counts.append(np.minimum(4, npg - 4 * gi))
            heads.append(np.full(ngr, h))
            cont.append(fl)
            tc.append(tcs)
            page += npg
        at.append((n, ngr))
        n += kvh * ngr
    cat = lambda v, t: torch.from_numpy(np.concatenate(v).astype(t)).to(DEV)  # noqa: E731
    return {"first": cat(first, np.int64), "counts": cat(counts, np.int32), "heads": cat(heads, np.int32),
            "cont": cat(cont, np.uint8), "tc": cat(tc, np.int32), "at": at, "groups": n, "pages": page - base}


def _tables(k, v, kvh):
    """One decode table per head for K and V, from a sample of the pages a program calibrated on."""
    out = []
    for h in range(kvh):
        for x in (k, v):
            out.append(kv.build_table(x[: 24 * kvh][h::kvh][:16].cpu().numpy()))
    return torch.from_numpy(np.concatenate(out)).to(DEV)


def _encode(codec, k, v, hd, tab, g, pool, at):
    r = kv.encode_groups_device(codec, k, v, hd, tab, g["first"], g["counts"], pool, at, g["heads"], g["tc"],
                                continues=g["cont"] if codec != kv.CODEC_INT8 else None)
    if int(r.status.item()) != 0:
        raise RuntimeError("sealing failed")
    return r


def _blob_max(codec, hd):
    return int(A.lib().cf_kv_group_blob_max_bytes(codec, hd))


def _prepare_decode(case, seed):
    lens, kvh, hd, S = _lens(case), case["kvh"], case["hd"], case["seqs"]
    codec = kv.CODEC_RANS_HYBRID if case.get("codec", "rans") == "rans" else kv.CODEC_INT8
    shared = case.get("shared", 0)
    sg = shared // 64
    mg = sg + max((t + 63) // 64 for t in lens)
    offs = torch.zeros((S, kvh, mg), dtype=torch.int32, device=DEV)
    g = _groups(lens, kvh, sg if shared else None)
    k, v = _kv_values(seed, g["pages"], hd)
    tab = _tables(k, v, kvh) if codec == kv.CODEC_RANS_HYBRID else None
    cap = g["groups"] * _blob_max(codec, hd) + (kvh * sg * _blob_max(kv.CODEC_INT8, hd) if shared else 0)
    big = torch.empty(cap + 16, dtype=torch.uint8, device=DEV)
    at = 0
    if shared:  # the prefix: one INT8 copy, named by every sequence
        pg = _groups([shared], kvh)
        pk, pv = _kv_values(seed, pg["pages"], hd, 1)
        r = _encode(kv.CODEC_INT8, pk, pv, hd, None, pg, big, 0)
        offs[:, :, :sg] = r.offsets.view(kvh, sg)
        at = int(r.pool_end.item())
        del pk, pv
    r = _encode(codec, k, v, hd, tab, g, big, at)
    del k, v
    for s, (n0, ngr) in enumerate(g["at"]):
        offs[s, :, sg:sg + ngr] = r.offsets[n0:n0 + kvh * ngr].view(kvh, ngr)
    pool = big[:int(r.pool_end.item())].clone()
    del big
    tok = torch.tensor([shared + t for t in lens], dtype=torch.int32, device=DEV)
    kvb = kv.BatchedKv(codec, S, kvh, hd, mg, pool, offs, tok, tab)
    q = torch.randn((S, kvh * case["gqa"], hd), generator=_gen(seed, 2), device=DEV)
    out = torch.empty_like(q)
    pos = tok - 1
    scale = 1.0 / math.sqrt(hd)
    desc = kvb.desc(q, out, pos, scale, 0, sg)
    return {"kv": kvb, "q": q, "out": out, "pos": pos, "scale": scale, "desc": desc, "sg": sg}


def _run_decode(s):
    s["kv"].attention(s["q"], s["out"], s["pos"], s["scale"], desc=s["desc"], shared_groups=s["sg"])
    return s["out"]


def _int8_pages(x, t):
    """Pages [h, pages, 16, d] as the 8-bit quantiser of the format keeps them (absmax / 127 per page, round half to
    even), in float64, [h, t, d]."""
    h, p, _, d = x.shape
    x = x.reshape(h, p * 16, d).clone()
    x[:, t:] = 0
    x = x.reshape(h, p, 16, d)
    s = _scale(x.abs().amax(dim=(2, 3), keepdim=True), 127.0)
    q = torch.clamp(torch.round(x / s), -128, 127)
    return (q.double() * s.double()).reshape(h, p * 16, d)[:, :t]


def _attend(q, k, v, scale):
    """q [h, g, d], k and v [h, t, d], all float64."""
    w = torch.softmax(torch.matmul(q, k.transpose(1, 2).contiguous()) * scale, dim=-1)
    return torch.matmul(w, v)


def _exact_decode(case, seed):
    lens, kvh, hd, S, gqa = _lens(case), case["kvh"], case["hd"], case["seqs"], case["gqa"]
    shared = case.get("shared", 0)
    npg = _pages_of(lens)
    k, v = _kv_values(seed, kvh * sum(npg), hd)
    q = torch.randn((S, kvh * gqa, hd), generator=_gen(seed, 2), device=DEV).double()
    if shared:
        pk, pv = (_int8_pages(x.view(kvh, shared // 16, 16, hd), shared) for x in _kv_values(seed, kvh * shared // 16, hd, 1))
    out = torch.empty_like(q)
    page = 0
    for s, t in enumerate(lens):
        ks, vs = (_int8_pages(x[page:page + kvh * npg[s]].view(kvh, npg[s], 16, hd), t) for x in (k, v))
        page += kvh * npg[s]
        if shared:
            ks, vs = torch.cat([pk, ks], 1), torch.cat([pv, vs], 1)
        out[s] = _attend(q[s].view(kvh, gqa, hd), ks, vs, 1.0 / math.sqrt(hd)).view(kvh * gqa, hd)
    return out


def _prepare_seal(case, seed):
    lens, kvh, hd = _lens(case), case["kvh"], case["hd"]
    codec = kv.CODEC_RANS_HYBRID if case["codec"] == "rans" else kv.CODEC_INT8
    g = _groups(lens, kvh)
    k, v = _kv_values(seed, g["pages"], hd)
    tab = _tables(k, v, kvh) if codec == kv.CODEC_RANS_HYBRID else None
    tcount = 2 * kvh if tab is not None else 0
    ws = torch.empty(int(A.lib().cf_kv_encode_groups_workspace_bytes(codec, hd, g["groups"], tcount)),
                     dtype=torch.uint8, device=DEV)
    pool = torch.zeros(g["groups"] * _blob_max(codec, hd), dtype=torch.uint8, device=DEV)
    return {"codec": codec, "k": k, "v": v, "hd": hd, "tab": tab, "g": g, "ws": ws, "pool": pool}


def _run_seal(s):
    g = s["g"]
    r = kv.encode_groups_device(s["codec"], s["k"], s["v"], s["hd"], s["tab"], g["first"], g["counts"], s["pool"], 0,
                                g["heads"], g["tc"], s["ws"],
                                continues=g["cont"] if s["codec"] != kv.CODEC_INT8 else None)
    return {"pool": s["pool"], "offsets": r.offsets, "end": r.pool_end, "status": r.status}


# ------------------------------------------------------------------------------------------------ coded int4 weights
def _weights(case, seed):
    """Weights N(0, 0.02) quantised to int4 per 64 columns of a row (absmax / 7): symbols q + 8 and scales."""
    rows, cols = case["rows"], case["cols"]
    ns = (cols + 63) // 64
    w = torch.zeros((rows, ns * 64), device=DEV)
    w[:, :cols] = 0.02 * torch.randn((rows, cols), generator=_gen(seed), device=DEV)
    w = w.view(rows, ns, 64)
    sc = _scale(w.abs().amax(dim=2), 7.0)
    q = torch.clamp(torch.round(w / sc[:, :, None]), -8, 7)
    return (q + 8).to(torch.uint8).view(rows, ns * 64)[:, :cols].contiguous(), sc


def _x(case, seed):
    return torch.randn((case["batch"], case["cols"]), generator=_gen(seed, 1), device=DEV).to(torch.bfloat16)


def _prepare_matmul(case, seed):
    sym, sc = _weights(case, seed)
    w = qw.QwMatrix(qw.encode_symbols(sym.cpu().numpy(), sc.cpu().numpy(), qw.QW_CODEC_RANS), DEV)
    return {"w": w, "x": _x(case, seed), "y": torch.empty((case["batch"], case["rows"]), device=DEV)}


def _run_matmul(s):
    s["w"].matmul_into(s["x"], s["y"])
    return s["y"]


def _exact_matmul(case, seed):
    sym, sc = _weights(case, seed)
    w = (sym.double() - 8.0) * sc.double().repeat_interleave(64, dim=1)[:, :case["cols"]]
    return torch.matmul(_x(case, seed).double(), w.t().contiguous())


# ------------------------------------------------------------------------------------------------ int4 nibble pages
_PAGE, _BLOCK = 64, 32


def _nib_items(case):
    """(tokens, query tokens) of each item: the first `chunks` are prefill chunks, the rest decode."""
    return [(max(t, case["chunk"]), case["chunk"]) if i < case["chunks"] else (t, 1) for i, t in enumerate(_lens(case))]


def _nib_kv(case, seed, i, t):
    return torch.randn((2, t, case["kvh"], case["hd"]), generator=_gen(seed, 10 + i), device=DEV)


def _nib_queries(case, seed):
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    g = _gen(seed, 3)
    return [torch.randn((n, case["kvh"] * case["gqa"], case["hd"]), generator=g, device=DEV).to(dt)
            for _, n in _nib_items(case)]


def _prepare_nibble(case, seed):
    items = _nib_items(case)
    H, QH, D = case["kvh"], case["kvh"] * case["gqa"], case["hd"]
    eng = sealkv.SealEngine(len(items), H, QH, D, _PAGE, _BLOCK)
    res = sealkv.MsResolver(1, H, QH, D, _PAGE)
    hold = []
    for i, (t, _) in enumerate(items):
        x = _nib_kv(case, seed, i, t)
        res.create(i)
        full = t // _PAGE
        for p in range(full):
            eng.stage(i, p * _PAGE, x[0, p * _PAGE:(p + 1) * _PAGE], x[1, p * _PAGE:(p + 1) * _PAGE])
            eng.seal(i)
        for d in eng.pages(i):
            res.publish(i, 0, d)
        if t % _PAGE:
            tail = x[:, full * _PAGE:].contiguous()
            hold.append(tail)
            res.stage_active(i, 0, full * _PAGE, tail[0], tail[1])
    q = _nib_queries(case, seed)
    out = [torch.empty_like(x) for x in q]
    sc = 1.0 / math.sqrt(D)
    arr = (sealkv.cf_ms_batch_item * len(items))()
    for i, (t, n) in enumerate(items):
        o = out[i]
        es = o.element_size()
        arr[i] = sealkv.cf_ms_batch_item(i, 0, sealkv.tensor_view(q[i]), o.data_ptr(),
                                         sealkv.CF_DEVICE_BF16 if case["dtype"] == "bf16" else sealkv.CF_DEVICE_F32,
                                         o.stride(0) * es, o.stride(1) * es, o.stride(2) * es, t - n, sc, 0)
    torch.cuda.synchronize()
    return {"res": res, "eng": eng, "q": q, "out": out, "arr": arr, "hold": hold}


def _run_nibble(s):
    L = A.lib()
    if L.cf_ms_cuda_execute_batch_async(s["res"].h, s["arr"], len(s["arr"]), torch.cuda.current_stream().cuda_stream) != 0:
        raise RuntimeError(L.cf_ms_cuda_last_error(s["res"].h).decode())
    return s["out"]


def _exact_nibble(case, seed):
    H, gqa, D = case["kvh"], case["gqa"], case["hd"]
    out = []
    for i, ((t, n), q) in enumerate(zip(_nib_items(case), _nib_queries(case, seed))):
        x = _nib_kv(case, seed, i, t)
        full = t // _PAGE * _PAGE
        b = x[:, :full].reshape(2, -1, _BLOCK)
        s = _scale(b.abs().amax(dim=2, keepdim=True), 7.0)
        d = torch.clamp(torch.round(b / s), -8, 7).double() * s.double()
        y = torch.cat([d.reshape(2, full, H, D), x[:, full:].double()], 1).permute(0, 2, 1, 3).contiguous()
        o = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for j in range(n):
            o[j] = _attend(q[j].double().view(H, gqa, D), y[0, :, :t - n + j + 1], y[1, :, :t - n + j + 1],
                           1.0 / math.sqrt(D)).view(H * gqa, D)
        out.append(o)
    return out


# ------------------------------------------------------------------------------------------------ the llama adapter
def _seam_inputs(case, seed):
    g = _gen(seed)
    x = torch.randn((2, case["kvh"], case["tokens"], case["hd"]), generator=g, device=DEV)
    q = torch.randn((min(case["queries"], case["tokens"]), case["kvh"] * case["gqa"], case["hd"]), generator=g, device=DEV)
    return x, q


def _prepare_seam(case, seed):
    x, q = _seam_inputs(case, seed)
    qh = case["kvh"] * case["gqa"]
    ad = llama.KvAdapter(llama.options(1, case["kvh"], qh, case["hd"], case["page"], case["gqa"], case["bits"]))
    host = x.cpu().numpy()
    for h in range(case["kvh"]):
        ad.append(0, h, 0, host[0, h], host[1, h])
    return {"ad": ad, "q": q, "out": torch.empty_like(q), "qh": qh, "gqa": case["gqa"],
            "begin": case["tokens"] - q.shape[0], "scale": 1.0 / math.sqrt(case["hd"])}


def _run_seam(s):
    q, out = s["q"], s["out"]
    s["ad"].attention(0, q.data_ptr(), out.data_ptr(), q.shape[0], s["qh"], s["gqa"], s["begin"], s["scale"], 0,
                      torch.cuda.current_stream().cuda_stream)
    return out


def _exact_seam(case, seed):
    x, q = _seam_inputs(case, seed)
    T, H, D, ps, top = case["tokens"], case["kvh"], case["hd"], case["page"], 2 ** (case["bits"] - 1)
    full = T // ps * ps
    p = x[:, :, :full].reshape(2, H, full // ps, ps, D)
    d = []
    for i, ax in ((0, 3), (1, 4)):  # K: one scale per channel of a page; V: one per token
        s = _scale(p[i:i + 1].abs().amax(dim=ax, keepdim=True), float(top - 1))
        d.append(torch.clamp(torch.round(p[i:i + 1] / s), -top, top - 1).double() * s.double())
    y = torch.cat([torch.cat(d).reshape(2, H, full, D), x[:, :, full:].double()], 2)
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    n = q.shape[0]
    for j in range(n):
        t = T - n + j + 1
        out[j] = _attend(q[j].double().view(H, case["gqa"], D), y[0, :, :t], y[1, :, :t],
                         1.0 / math.sqrt(D)).view(H * case["gqa"], D)
    return out


# ------------------------------------------------------------------------------------------------ compressed-domain search
_VOCAB, _SA_SAMPLE = 32000, 32


def _zipf(n, g):
    """Zipf(1.1) tokens over the vocabulary, by inverse-CDF sampling."""
    cdf = torch.cumsum(torch.arange(1, _VOCAB + 1, dtype=torch.float64, device=DEV) ** -1.1, 0)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_(max=_VOCAB - 1).to(torch.int32)


def _pattern_lens(case):
    r = np.random.default_rng(case["patterns"] + 31 * case["lmax"])
    return r.integers(case["lmin"], case["lmax"] + 1, case["patterns"])


def _prepare_search(case, seed):
    g = _gen(seed)
    tokens = _zipf(case["n"], g)
    fm, _ = search.build_fm(tokens, _SA_SAMPLE)
    fm.build_quads()
    # nine patterns in ten are cut from the text, one is random (almost never there)
    n, P = case["n"], case["patterns"]
    lens = torch.from_numpy(_pattern_lens(case)).to(DEV)
    start = torch.cumsum(lens, 0) - lens
    total = int(lens.sum().item())
    at = (torch.rand(P, generator=g, device=DEV, dtype=torch.float64) * (n - case["lmax"])).long()
    who = torch.repeat_interleave(torch.arange(P, device=DEV), lens)
    pat = tokens[at[who] + torch.arange(total, device=DEV) - start[who]] + 1
    rnd = torch.randint(1, _VOCAB + 1, (total,), generator=g, device=DEV, dtype=torch.int32)
    pat = torch.where(who % 10 == 9, rnd, pat).to(torch.int32)
    return {"fm": fm, "pat": pat, "start": start.to(torch.int32), "len": lens.to(torch.int32)}


def _run_search(s):
    fm = s["fm"]
    lo, hi = fm.ranges_quads(s["pat"], s["start"], s["len"])
    first = fm.locate_quads(torch.clamp(lo, max=fm.n - 1))
    return {"lo": lo, "hi": hi, "first": first}


def _prepare_wavelet(case, seed):
    g = _gen(seed)
    n, nq = case["n"], case["queries"]
    tokens = _zipf(n, g)
    idx, _ = search.build_rrrw(tokens, 15)
    idx.build_quads(n)
    pos = torch.randint(0, n, (nq,), generator=g, device=DEV, dtype=torch.int32)
    sym = torch.where(torch.arange(nq, device=DEV) % 2 == 0,  # half of the ranked symbols from the stream
                      tokens[torch.randint(0, n, (nq,), generator=g, device=DEV)],
                      torch.randint(0, _VOCAB, (nq,), generator=g, device=DEV, dtype=torch.int32)).to(torch.int32)
    upto = torch.randint(0, n + 1, (nq,), generator=g, device=DEV, dtype=torch.int32)
    return {"idx": idx, "tokens": tokens, "pos": pos, "sym": sym, "upto": upto, "access": torch.empty_like(pos),
            "rank": torch.empty_like(pos)}


def _run_wavelet(s):
    s["idx"].access_quads_into(s["pos"], s["access"])
    s["idx"].rank_quads_into(s["sym"], s["upto"], s["rank"])
    return {"access": s["access"], "rank": s["rank"]}


# ------------------------------------------------------------------------------------------------ the interface
_PREPARE = {"decode": _prepare_decode, "cascade": _prepare_decode, "seal": _prepare_seal, "matmul": _prepare_matmul,
            "nibble": _prepare_nibble, "seam": _prepare_seam, "search": _prepare_search, "wavelet": _prepare_wavelet}
_RUN = {"decode": _run_decode, "cascade": _run_decode, "seal": _run_seal, "matmul": _run_matmul, "nibble": _run_nibble,
        "seam": _run_seam, "search": _run_search, "wavelet": _run_wavelet}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    f = {"decode": _exact_decode, "cascade": _exact_decode, "matmul": _exact_matmul, "nibble": _exact_nibble,
         "seam": _exact_seam}.get(case["kind"])
    return f(case, seed) if f else None  # the others return bytes and whole numbers


def work(case):
    kind = case["kind"]
    if kind in ("decode", "cascade"):
        per = 7.4 / 8 if case.get("codec", "rans") == "rans" else 1.0  # bytes per coded value, headers aside
        T, H, D = sum(_lens(case)), case["kvh"], case["hd"]
        shared = case.get("shared", 0)
        qo = 2 * 4 * case["seqs"] * H * case["gqa"] * D
        return {"bytes": 2 * H * D * (T * per + shared) + qo,
                "flops": 4.0 * H * case["gqa"] * D * (T + case["seqs"] * shared)}
    if kind == "seal":
        v = 2 * case["kvh"] * case["hd"] * sum(_lens(case))
        return {"bytes": v * (4 + (7.4 / 8 if case["codec"] == "rans" else 1.0)), "flops": 3.0 * v}
    if kind == "matmul":
        m, k, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": m * k * 4.25 / 8 + 2 * b * k + 4 * b * m, "flops": 2.0 * m * k * b}
    if kind == "nibble":
        H, D, G = case["kvh"], case["hd"], case["gqa"]
        es = 2 if case["dtype"] == "bf16" else 4
        items = _nib_items(case)
        by = sum(t // _PAGE * _PAGE * 2 * H * D * (0.5 + 4 / _BLOCK) + t % _PAGE * 2 * H * D * 4 + 2 * n * H * G * D * es
                 for t, n in items)
        return {"bytes": by, "flops": 4.0 * H * G * D * sum(t * n for t, n in items)}
    if kind == "seam":
        T, H, D = case["tokens"], case["kvh"], case["hd"]
        n = min(case["queries"], T)
        return {"bytes": 2 * H * D * T * case["bits"] / 8 + 2 * 4 * n * H * case["gqa"] * D,
                "flops": 4.0 * n * H * case["gqa"] * D * T}
    if kind == "search":
        # per pattern symbol two walks of 8 records of 64 bytes; per located row half a sample period of walks
        s, p = float(_pattern_lens(case).sum()), case["patterns"]
        return {"bytes": s * (2 * 8 * 64 + 4) + p * (_SA_SAMPLE / 2 * 8 * 64 + 16), "flops": 0.0}
    return {"bytes": case["queries"] * (2 * 8 * 64 + 20), "flops": 0.0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("seal", "search", "wavelet"):
        return "exact"
    if kind == "nibble" and case["dtype"] == "bf16":
        return {"rel": 4e-3, "max": 3e-2}  # outputs rounded to bf16
    if kind == "matmul":
        return {"rel": 1e-6, "max": 2e-5}  # exact products, float32 sums: 1e-7 off
    if kind == "decode":
        return {"rel": 2e-5}  # the longest contexts are 5e-6 off (f16 hi + lo operands, a running maximum per wavefront)
    return {"rel": 4e-6}  # the same operands, shorter sums: 6e-7 off
