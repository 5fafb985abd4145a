"""The device encoder's arithmetic where it differs from the host's: quotients by a reciprocal (exact division near a
rounding boundary, for non-finite values and extreme scales) and the coder's division by a multiplication. Bytes against
the host encoder cf_kv_encode_groups on pages whose quotients lie on and one or a few ulps beside n + 1/2, on scales from
denormal to the largest, on negative zeros, and on -128 beside coded groups."""
import numpy as np
import pytest


def test_coder_division_is_exact():
    """mulhi(x, floor(2^32 / f)) with one correction is x / f, x % f for every frequency and states at the edges of its
    quotients."""
    f = np.arange(2, 2048, dtype=np.uint64)[:, None]
    k = np.array([1, 2, 3, 1000, 2 ** 20, 2 ** 21 - 1], np.uint64)[None, :]
    x = np.concatenate([np.minimum(f * k + d, 2 ** 32 - 1) for d in (0, 1)] + [f * k - 1] +
                       [np.broadcast_to(np.array([2 ** 32 - 1, 2 ** 31, 2 ** 16], np.uint64), (f.size, 3))], axis=1)
    x = np.minimum(x, 2 ** 32 - 1).astype(np.uint64)
    q = (x * (2 ** 32 // f)) >> np.uint64(32)
    r = x - q * f
    assert ((r < 2 * f) & (r < 2 ** 32)).all()
    q, r = np.where(r >= f, q + 1, q), np.where(r >= f, r - f, r)
    assert np.array_equal(q, x // f) and np.array_equal(r, x % f)


@pytest.mark.gpu
@pytest.mark.parametrize("codec", ["rans", "int8"])
@pytest.mark.parametrize("D", [64, 96, 128])
def test_rounding_boundaries(codec, D):
    import torch
    from chromofold_amd import kv
    print(f"case {codec} D={D}", flush=True)
    cdc = kv.CODEC_RANS_HYBRID if codec == "rans" else kv.CODEC_INT8
    rng = np.random.default_rng(D)
    pages = []
    for top in (127.0, 1.0, 3.7e-5, 1e-37, 2e-39, 1.2e-44, 3e37, 1e-31, 1.3e32):
        with np.errstate(all="ignore"):
            s = np.float32(top) / np.float32(127)
            n = rng.integers(-127, 127, (16, D)).astype(np.float32) + np.float32(0.5)
            x = (n.astype(np.float64) * s).astype(np.float32)
            for _ in range(3):  # up to three ulps to either side
                step = rng.integers(-1, 2, x.shape)
                x = np.where(step < 0, np.nextafter(x, np.float32(-np.inf)), np.where(step > 0, np.nextafter(x, np.float32(np.inf)), x))
        x[0, 0] = top
        x[1, :4] = [0.0, -0.0, np.float32(s) * np.float32(0.25), -np.float32(s) * np.float32(0.25)]
        pages.append(x.astype(np.float32))
    odd = rng.standard_normal((3, 16, D)).astype(np.float32)
    odd[0, 2, 3], odd[1, 4, 5], odd[2, 6, 7] = np.nan, np.inf, -np.inf
    K = np.stack(pages + list(odd) + [np.zeros((16, D), np.float32)] * 3)  # 15 pages
    V = K[::-1].copy()
    first = np.arange(0, 15, 3).astype(np.uint64)  # five groups of three pages, in chain pairs
    counts = np.full(5, 3, np.uint32)
    cont = np.array([0, 1, 0, 1, 0], np.uint8)
    tc = np.array([16, 16, 5] * 5, np.uint32)
    tables = np.concatenate([kv.build_table(rng.standard_normal((4, 16, D)).astype(np.float32)) for _ in range(2)])
    tables = tables if codec == "rans" else None
    args = dict(continues=cont if codec == "rans" else None)
    with np.errstate(all="ignore"):
        want, offs = kv.encode_groups(cdc, K, V, D, tables, first, counts, None, tc, **args)
    up = lambda a, t=None: None if a is None else torch.from_numpy(a if t is None else a.astype(t)).to("cuda:0")  # noqa: E731
    pool = torch.zeros(want.size + 4096, dtype=torch.uint8, device="cuda:0")
    r = kv.encode_groups_device(cdc, up(K), up(V), D, up(tables), up(first, np.int64), up(counts, np.int32), pool, 0, None,
                                up(tc, np.int32), continues=up(cont) if codec == "rans" else None)
    torch.cuda.synchronize()
    assert int(r.status.item()) == 0 and int(r.pool_end.item()) == want.size
    assert np.array_equal(r.offsets.cpu().numpy().view(np.uint32), offs)
    assert np.array_equal(pool.cpu().numpy()[:want.size], want)


@pytest.mark.gpu
@pytest.mark.parametrize("codec", ["rans", "int8"])
@pytest.mark.parametrize("D", [64, 96, 128])
def test_scale_zero_pages_with_absent_tokens(codec, D):
    """An absmax below 64 of the smallest denormals gives a scale of 0: present values become -128 (their quotients are
    infinite or no number), absent tokens stay 0, whatever the page's token count leaves of the last four tokens."""
    import torch
    from chromofold_amd import kv
    print(f"case {codec} D={D}", flush=True)
    cdc = kv.CODEC_RANS_HYBRID if codec == "rans" else kv.CODEC_INT8
    rng = np.random.default_rng(D)
    tc = np.array([1, 2, 3, 4, 5, 7, 9, 11, 13, 14, 15, 16, 6, 10, 12, 8], np.uint32)
    tiny = rng.integers(-63, 64, (16, 16, D)).astype(np.float64) * 2.0 ** -149
    tiny[:, 0, 0] = 63 * 2.0 ** -149
    V = tiny.astype(np.float32)
    K = rng.standard_normal((16, 16, D)).astype(np.float32)
    K[8:] = V[:8]
    tables = np.concatenate([kv.build_table(rng.standard_normal((4, 16, D)).astype(np.float32)) for _ in range(2)])
    tables = tables if codec == "rans" else None
    first, counts = np.arange(0, 16, 4).astype(np.uint64), np.full(4, 4, np.uint32)
    with np.errstate(all="ignore"):
        want, offs = kv.encode_groups(cdc, K, V, D, tables, first, counts, None, tc)
    up = lambda a, t=None: None if a is None else torch.from_numpy(a if t is None else a.astype(t)).to("cuda:0")  # noqa: E731
    pool = torch.zeros(want.size + 4096, dtype=torch.uint8, device="cuda:0")
    r = kv.encode_groups_device(cdc, up(K), up(V), D, up(tables), up(first, np.int64), up(counts, np.int32), pool, 0, None,
                                up(tc, np.int32))
    torch.cuda.synchronize()
    assert int(r.status.item()) == 0 and int(r.pool_end.item()) == want.size
    assert np.array_equal(r.offsets.cpu().numpy().view(np.uint32), offs)
    assert np.array_equal(pool.cpu().numpy()[:want.size], want)
