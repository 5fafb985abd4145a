"""Mixed batches over int4 nibble pages: items of different context lengths, query-token counts and tails in one call
(cf_ms_cuda_execute_batch_async), every item against the oracle's float64 attention over the same pages (semantics of
reference src/cuda/multisequence_cuda_resolver.cu:136-195).

Sizes sit where the launches can go wrong: items that own no workgroup of a launch (no sealed page, no tail, neither)
beside ones that own many, more than 64 items, tails around the tokens of one split (8) and of a whole page, query
chunks that are no multiple of the query tokens a workgroup takes, a window that hides whole pages.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kvh,gqa,D,page,bs", [(2, 4, 128, 64, 32),    # matrix-core kernel, four scale blocks a row
                                               (3, 3, 128, 48, 64),    # two blocks, a ragged last chunk
                                               (1, 5, 128, 32, 128),   # one block, two chunks of query heads
                                               (2, 2, 64, 16, 32)])    # VALU kernel
@pytest.mark.parametrize("copies", [1, 5])
def test_mixed_batch(kvh, gqa, D, page, bs, copies):
    import torch
    from chromofold_amd.sealkv import MsResolver, SealEngine
    dev = torch.device("cuda:0")
    print(f"case kvh={kvh} gqa={gqa} D={D} page={page} bs={bs} copies={copies}", flush=True)
    rng = np.random.default_rng(page + D + copies)
    qh = kvh * gqa
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    # (pages, tail tokens, query tokens, window)
    shapes = [(0, 0, 1, 0), (0, 1, 1, 0), (3, 0, 1, 0), (0, 7, 4, 0), (5, 8, 1, 0), (1, 9, 9, 0), (11, page - 1, 3, 0),
              (2, 16, 2, 0), (4, 3, 5, 2 * page), (7, 0, 7, 5), (1, 0, 16, 0), (0, 0, 2, 0), (9, 4, 1, page)]
    eng = SealEngine(len(shapes), kvh, qh, D, page, bs)
    res = MsResolver(1, kvh, qh, D, page)
    state = []
    for s, (np_, tail, _, _) in enumerate(shapes):
        res.create(s)
        pages = []
        for p in range(np_):
            k, v = (rng.standard_normal((page, kvh, D)).astype(np.float32) for _ in range(2))
            eng.stage(s, p * page, up(k), up(v))
            eng.seal(s)
            pages.append(O.nib_seal_page(k, v, p * page, bs))
        for d in eng.pages(s):
            res.publish(s, 0, d)
        ak = av = None
        if tail:
            ak, av = (rng.standard_normal((tail, kvh, D)).astype(np.float32) for _ in range(2))
            res.stage_active(s, 0, np_ * page, up(ak), up(av))
        state.append((pages, ak, av))
    items, refs = [], []
    for c in range(copies):
        for s, (np_, tail, qt, window) in enumerate(shapes):
            total = np_ * page + tail
            begin = max(0, total - qt) if c % 2 == 0 else max(0, total // 2 - qt)  # at the end, and mid-context
            q = rng.standard_normal((qt, qh, D)).astype(np.float32)
            out = torch.full((qt, qh, D), float("nan"), device=dev)
            items.append((s, 0, up(q), out, begin, 0.09, window))
            pages, ak, av = state[s]
            refs.append(O.nib_attention(pages, bs, q, begin, kvh, gqa, 0.09, window, ak, av, np_ * page)
                        if pages or ak is not None else np.zeros_like(q))
    res.execute(items)
    torch.cuda.synchronize()
    for i, ((s, _, _, out, begin, _, _), ref) in enumerate(zip(items, refs)):
        got = out.cpu().numpy()
        assert np.isfinite(got).all(), (i, shapes[s])
        # f16 hi + lo operands (2^-21 per product) and fp32 sums: 2e-6 of the row's norm is typical, 2e-5 the bound
        err = np.linalg.norm(got - ref, axis=-1) / np.maximum(np.linalg.norm(ref, axis=-1), 1e-3)
        assert err.max() <= 2e-5, (i, shapes[s], begin, float(err.max()))
    res.reclaim()
    res.close()
    eng.close()
