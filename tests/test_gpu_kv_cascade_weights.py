"""Small softmax weights in the cascade's prefix pass: rows whose heavy tokens have V = 0 and whose output comes from tokens
of 2^-20 to 2^-24 of the largest weight, with V scales that fall after a first, even lighter group of larger ones. Against
a float64 softmax over the quantised pages."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("drop", [2.0, 4.0, 16.0])
@pytest.mark.parametrize("bits", [20, 22, 24])
def test_light_tokens_carry_the_row(bits, drop):
    """Every prefix split sees the same three kinds of groups: heavy ones, lighter ones with V `drop` times larger than the
    rest's, then the tokens of weight 2^-bits that carry the row."""
    import torch
    from chromofold_amd import kv
    print(f"case bits={bits} drop={drop}", flush=True)
    dev, D, H, S, shared = torch.device("cuda:0"), 128, 2, 128, 128
    n = 64 * shared
    rng = np.random.default_rng(bits)
    k = np.zeros((H, n + 1, D), np.float32)
    v = rng.standard_normal((H, n + 1, D)).astype(np.float32)
    v /= np.abs(v).max() / 3
    k[:, :, 1:] = 0.01 * rng.standard_normal((H, n + 1, D - 1))
    per = shared // 32  # of a split: 2 * 256 CUs / (2 heads * 8 row tiles) = 32 splits
    gap = bits * np.log(2.0)
    for g in range(shared):
        t = slice(64 * g, 64 * g + 64)
        kind = g % per
        k[:, t, 0] = gap / 2 if kind == 0 else -gap / 2 - 6 * np.log(2.0) if kind == 1 else -gap / 2
        v[:, t] *= 0.0 if kind == 0 else drop if kind == 1 else 1.0
    k[:, -1, 0], v[:, -1] = -40.0, 0.0  # the one own token weighs nothing
    tables = np.concatenate([kv.build_table(x[h][:256].reshape(-1, 16, D)) for h in range(H) for x in (k, v)])
    kvb = kv.build_batched(kv.CODEC_RANS_HYBRID, lambda s: (k, v), S, H, np.full(S, n + 1), D, tables, dev,
                           shared={s: (0, shared) for s in range(1, S)}, raw_groups={0: shared})
    q = np.zeros((S, H, D), np.float32)
    q[:, :, 0] = 1.0 + 0.01 * rng.random((S, H))
    q[:, :, 1:] = 0.2 * rng.standard_normal((S, H, D - 1))
    dq = torch.from_numpy(q).to(dev)
    out = torch.full_like(dq, float("nan"))
    pos = torch.full((S,), n, dtype=torch.int32, device=dev)
    d = kvb.desc(dq, out, pos, 1.0, 1, shared)
    assert d.workspace_bytes == S * H * (32 + 1) * 4 * (D + 2) * 4, "32 prefix splits"
    kvb.attention(dq, out, pos, 1.0, desc=d, shared_groups=shared)
    got = out.cpu().double()

    def deq(x):
        x = torch.from_numpy(x[:, :n]).view(H, -1, 16, D)
        m = x.abs().amax(dim=(2, 3), keepdim=True)
        s = torch.where(m == 0, torch.ones_like(m), m / 127.0)
        return (torch.round(x / s).double() * s.double()).view(H, -1, D)

    kq, vq = deq(k), deq(v)
    qd = torch.from_numpy(q).double()
    err = 0.0
    for h in range(H):
        want = torch.matmul(torch.softmax(torch.matmul(qd[:, h], kq[h].t().contiguous()), -1), vq[h])
        err = max(err, float(((got[:, h] - want).norm(dim=-1) / want.norm(dim=-1)).max()))
    # A weight's f16 parts keep it to 2^-25 of its unit (f16 subnormals), in which one of 2^-bits of the largest lies at or
    # above 2^(14 - bits): 2^(bits - 39) of it. The lighter group's weights are kept to the same 2^-25 beside V `drop` times
    # as large. Scores, exponents of up to 12 in float32 from 22-bit operands, are off by up to 2^-19, twice for the sum.
    bound = 2.0 ** (bits - 39) * (1 + drop) + 2.0 ** -18
    print(f"error {err:.2e} bound {bound:.2e}", flush=True)
    assert err <= bound
