"""The unit of the matrix-core nibble kernel's weights (p * v_scale as f16 hi + lo in units that follow the largest V scale
met so far): V magnitudes far below and above 1, rising and falling from page to page, all-zero pages, tails whose values
are far above the pages' or near the largest float. Against the oracle's float64 attention over the same pages."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [32, 64, 128])
def test_v_magnitudes(bs):
    import torch
    from chromofold_amd.sealkv import MsResolver, SealEngine
    dev, kvh, gqa, page, D = torch.device("cuda:0"), 2, 4, 64, 128
    print(f"case bs={bs}", flush=True)
    rng = np.random.default_rng(bs)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    # (V magnitude of each page, tail tokens, V magnitude of the tail)
    shapes = [([1.0] * 33, 0, 1), ([1e-6] * 5, 0, 1), ([1e6] * 5, 0, 1), ([1e-25] * 3, 0, 1), ([1e30] * 3, 5, 1e30),
              (list(10.0 ** np.arange(-8, 9)), 0, 1), (list(10.0 ** np.arange(8, -9, -1)), 0, 1),
              ([0.0, 1e-4, 0.0, 3.0, 0.0], 0, 1), ([1e-5, 1e5] * 20, 0, 1), ([1.0] * 9, 20, 1.0), ([1e-6] * 9, 20, 1e-6),
              ([1e-3] * 5, 17, 1e6), ([1e6] * 5, 63, 1e-3), ([1.0] * 5, 5, 2e37), ([0.0], 3, 1.0)]
    eng = SealEngine(len(shapes), kvh, kvh * gqa, D, page, bs)
    res = MsResolver(1, kvh, kvh * gqa, D, page)
    items, refs = [], []
    for s, (mags, tail, tm) in enumerate(shapes):
        res.create(s)
        sealed = []
        for p, mag in enumerate(mags):
            k, v = (rng.standard_normal((page, kvh, D)).astype(np.float32) for _ in range(2))
            v *= np.float32(mag)
            eng.stage(s, p * page, up(k), up(v))
            eng.seal(s)
            sealed.append(O.nib_seal_page(k, v, p * page, bs))
        for d in eng.pages(s):
            res.publish(s, 0, d)
        ak = av = None
        if tail:
            ak, av = (rng.standard_normal((tail, kvh, D)).astype(np.float32) for _ in range(2))
            av *= np.float32(tm)
            res.stage_active(s, 0, len(mags) * page, up(ak), up(av))
        total = len(mags) * page + tail
        q = rng.standard_normal((2, kvh * gqa, D)).astype(np.float32)
        out = torch.full(q.shape, float("nan"), device=dev)
        items.append((s, 0, up(q), out, total - 2, 0.09, 0))
        refs.append(O.nib_attention(sealed, bs, q, total - 2, kvh, gqa, 0.09, 0, ak, av, len(mags) * page))
    res.execute(items)
    torch.cuda.synchronize()
    for shape, (_, _, _, out, _, _, _), ref in zip(shapes, items, refs):
        got = out.cpu().numpy().astype(np.float64)
        ref = ref.astype(np.float64)
        assert np.isfinite(got).all(), shape
        # weights of 22 bits and float32 sums: 2.5e-7 of a row is typical, 2^-19 eight times that
        err = np.linalg.norm(got - ref, axis=-1) / np.maximum(np.linalg.norm(ref, axis=-1), 1e-37)
        assert err.max() <= 2.0 ** -19, (shape[0][:3], shape[1:], float(err.max()))
    res.reclaim()
    res.close()
    eng.close()


@pytest.mark.parametrize("mode", ["resolver32", "resolver64", "resolver128", "runtime"])
def test_negative_v_scales(mode):
    """Pages a caller publishes with scales of its own: V scales of either sign and of several magnitudes, all of them
    negative among others."""
    import torch
    from chromofold_amd import sealkv as S
    dev, kvh, gqa, page, D = torch.device("cuda:0"), 2, 4, 32, 128
    print(f"case {mode}", flush=True)
    rng = np.random.default_rng(11)
    keep = []

    def up(a):
        keep.append(torch.from_numpy(np.ascontiguousarray(a)).to(dev))
        return keep[-1]

    flips = [lambda v: -np.abs(v), lambda v: np.where(rng.random(v.shape) < 0.5, -v, v).astype(np.float32)]
    mags = [[1.0] * 5, [1e-3] * 33, [1e3] * 5, [1e4, 1e-4] * 4]
    q = rng.standard_normal((1, kvh * gqa, D)).astype(np.float32)
    outs, refs = [], []
    if mode == "runtime":
        bs = 32
        rt = S.AttentionRuntime(1, kvh, kvh * gqa, D, gqa=gqa, page_size=page, block_size=bs)
        items = (S.cf_attention_batch_item * (len(flips) * len(mags)))()
    else:
        bs = int(mode[8:])
        res, batch = S.MsResolver(1, kvh, kvh * gqa, D, page), []
    for i, (flip, mag) in enumerate((f, m) for f in flips for m in mags):
        descs, host = (S.cf_device_page_descriptor * len(mag))(), []
        for p, amp in enumerate(mag):
            k, v = (rng.standard_normal((page, kvh, D)).astype(np.float32) for _ in range(2))
            v *= np.float32(amp)
            if mode == "runtime":
                (kp, ks), (vp, vs) = O.rt_quantize(k, bs), O.rt_quantize(v, bs)
                vs = flip(vs)
                host.append(O.RtPage(kp, vp, ks, vs, p * page, page, D, bs))
            else:
                s = O.nib_seal_page(k, v, p * page, bs)
                kp, ks, vp, vs = s.k_payload, s.k_scales, s.v_payload, flip(s.v_scales)
                host.append(O.NibPage(kp, vp, ks, vs, p * page, page))
            d = descs[p]
            d.key_payload, d.value_payload, d.key_scales, d.value_scales = (up(a).data_ptr() for a in (kp, vp, ks, vs))
            d.token_begin, d.token_count, d.kv_head_count, d.head_dim, d.block_size = p * page, page, kvh, D, bs
        qpos, out = len(mag) * page - 1, torch.full((1, kvh * gqa, D), float("nan"), device=dev)
        outs.append(out)
        if mode == "runtime":
            it, qd = items[i], up(q)
            it.sequence_id, it.layer = 100 + i, 0
            it.query = S.cf_device_tensor_view(qd.data_ptr(), S._TYPE[qd.dtype], 1, kvh * gqa, D, 0, 4 * D, 4, 0)
            it.output, it.output_type = out.data_ptr(), S._TYPE[out.dtype]
            it.output_token_stride_bytes, it.output_head_stride_bytes, it.output_element_stride_bytes = 0, 4 * D, 4
            it.query_token_begin, it.softmax_scale, it.causal_window = qpos, 0.09, 0
            it.sealed_pages = up(np.frombuffer(bytearray(descs), np.uint8)).data_ptr()
            it.sealed_page_count = len(mag)
            refs.append(O.rt_attention_f64(q[0], kvh, gqa, qpos, 0, it.softmax_scale, host, None, None, 0))
        else:
            res.create(i)
            for d in descs:
                res.publish(i, 0, d)
            batch.append((i, 0, up(q), out, qpos, 0.09, 0))
            refs.append(O.nib_attention(host, bs, q, qpos, kvh, gqa, 0.09, 0))
    rt.execute(items) if mode == "runtime" else res.execute(batch)
    torch.cuda.synchronize()
    for i, (out, ref) in enumerate(zip(outs, refs)):
        got, ref = out.cpu().numpy().astype(np.float64).reshape(-1, D), ref.astype(np.float64).reshape(-1, D)
        assert np.isfinite(got).all(), i
        err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
        assert err.max() <= 2.0 ** -19, (i, float(err.max()))
    rt.close() if mode == "runtime" else (res.reclaim(), res.close())
