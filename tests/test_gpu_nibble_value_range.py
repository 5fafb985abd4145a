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
