"""Scores of -inf and NaN in the fp32 tail of an int4 sequence (its values are not checked when they are staged): a token
that scores -inf has no weight wherever it stands, first of a lane row's tokens included; a score that is no number makes
the rows that see it NaN. On both kernels that read tails (head_dim 128: matrix cores, 64: VALU), against the oracle's
float64 attention."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,bs", [(128, 32), (128, 64), (128, 128), (64, 32)])
@pytest.mark.parametrize("pages", [0, 1, 5])
def test_unusual_scores_in_the_tail(D, bs, pages):
    import torch
    from chromofold_amd.sealkv import MsResolver, SealEngine
    dev, kvh, gqa, page = torch.device("cuda:0"), 2, 4, 32
    print(f"case D={D} bs={bs} pages={pages}", flush=True)
    rng = np.random.default_rng(D + bs + pages)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    # (tail tokens, those that score -inf, those that score NaN)
    tails = [(1, [0], []), (2, [0], []), (9, [0, 1, 2, 3], []), (17, [0], []), (17, [0, 16], []), (31, list(range(30)), []),
             (31, list(range(0, 31, 2)), []), (20, list(range(20)), []), (5, [], [4]), (20, [3], [0, 1, 2]), (31, [], [30])]
    eng = SealEngine(len(tails), kvh, kvh * gqa, D, page, bs)
    res = MsResolver(1, kvh, kvh * gqa, D, page)
    items, refs = [], []
    for s, (n, low, nan) in enumerate(tails):
        res.create(s)
        sealed = []
        for p in range(pages):
            k, v = (rng.standard_normal((page, kvh, D)).astype(np.float32) for _ in range(2))
            eng.stage(s, p * page, up(k), up(v))
            eng.seal(s)
            sealed.append(O.nib_seal_page(k, v, p * page, bs))
        for d in eng.pages(s):
            res.publish(s, 0, d)
        ak, av = (rng.standard_normal((n, kvh, D)).astype(np.float32) for _ in range(2))
        q = rng.standard_normal((3, kvh * gqa, D)).astype(np.float32)
        q[:, :, 0] = np.abs(q[:, :, 0]) + 0.1
        ak[low, :, 0] = -np.inf
        ak[nan, :, 1] = np.nan
        res.stage_active(s, 0, pages * page, up(ak), up(av))
        out = torch.full(q.shape, 5.0, device=dev)
        begin = pages * page + n - 1  # every query sees the whole tail
        items.append((s, 0, up(q), out, begin, 0.09, 0))
        # the oracle without the tokens that have no weight
        keep = [t for t in range(n) if t not in low]
        kf, vf = np.where(np.isfinite(ak), ak, 0)[keep], av[keep]
        ref = (O.nib_attention(sealed, bs, q, begin, kvh, gqa, 0.09, 0, kf if keep else None, vf if keep else None,
                               pages * page) if sealed or keep else np.zeros_like(q))
        refs.append(np.full_like(q, np.nan) if nan else ref)
    res.execute(items)
    torch.cuda.synchronize()
    for (n, low, nan), (_, _, _, out, _, _, _), ref in zip(tails, items, refs):
        got = out.cpu().numpy()
        if nan:
            assert np.isnan(got).all(), (n, low, nan)
            continue
        assert np.isfinite(got).all(), (n, low)
        err = np.linalg.norm(got - ref, axis=-1) / np.maximum(np.linalg.norm(ref, axis=-1), 1e-3)
        assert err.max() <= 2e-5, (n, low, float(err.max()))  # the bound of the mixed batches' test
    res.reclaim()
    res.close()
    eng.close()
