"""The cascade's prefix pass (cf_kv_paged_attention_cascade_async) where its softmax reference and its V units move:
scores that rise over the groups by less and by more than ln 2, V magnitudes that rise and fall by fewer and more binary
exponents than the units follow, all-zero V pages, queries that end inside the prefix, row tiles of 1 to 33 sequences,
(head, split) units that are no multiple of the eight XCDs, prefix splits of one group and of several. splits = 1 takes
the rows that one workgroup finishes together with the prefix states, splits = 3 the merge launch. Against a float64
softmax over the quantised pages in torch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dequant(x):
    import torch
    H, T, D = x.shape
    x = torch.from_numpy(np.pad(x, ((0, 0), (0, (-T) % 16), (0, 0)))).view(H, -1, 16, D)
    m = x.abs().amax(dim=(2, 3), keepdim=True)
    s = torch.where(m == 0, torch.ones_like(m), m / 127.0)
    return (torch.round(x / s).double() * s.double()).view(H, -1, D)[:, :T]


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("H,gqa,shared,S", [(8, 4, 8, 5), (3, 2, 13, 17), (1, 3, 40, 33), (5, 1, 5, 16), (2, 4, 70, 1)])
def test_prefix_pass_against_float64(H, gqa, shared, S, splits):
    _check(H, gqa, shared, S, splits, [1, 17, 64, 200])


@pytest.mark.parametrize("shared", [1, 7, 8, 9])
@pytest.mark.parametrize("own", [[1, 200], [3100, 3300]])
def test_prefix_states_of_one_workgroup(shared, own):
    """Rows of one workgroup with as many prefix states as it adds itself (1 to 8, one per group here) and one more, which
    takes the merge launch; 4 wavefronts per workgroup, and 12."""
    _check(2, 3, shared, 5, 1, own)


def _check(H, gqa, shared, S, splits, own_lens):
    import torch
    from chromofold_amd import kv
    print(f"case H={H} gqa={gqa} shared={shared} S={S} splits={splits}", flush=True)
    dev, D, n = torch.device("cuda:0"), 128, 64 * shared
    rng = np.random.default_rng(100 * H + shared)
    q = rng.standard_normal((S, H * gqa, D)).astype(np.float32)
    common = rng.standard_normal((H, D)).astype(np.float32)
    q += 0.3 * np.repeat(common, gqa, 0)  # the ramp of the keys along `common` raises every row's scores
    lens = [n + int(rng.choice(own_lens)) for _ in range(S)]
    pos = [t - 1 for t in lens]
    pos[S // 2] = n // 2 + 5  # inside the prefix
    pos[-1] = lens[-1] - 1 if S > 1 else n - 64
    ramp = np.repeat(np.cumsum(rng.choice([0.0, 0.2, 1.5], shared)), 64) / 40
    vexp = np.repeat(rng.choice([-9, -1, 0, 1, 2, 3, 8], shared), 64).astype(np.float32)
    k0 = rng.standard_normal((H, n, D)).astype(np.float32) + (ramp[:, None] * common[:, None, :]).astype(np.float32)
    v0 = rng.standard_normal((H, n, D)).astype(np.float32) * np.exp2(vexp)[:, None]
    v0[:, 64:128] = 0.0  # (nothing where the prefix is one group)
    data = []
    for T in lens:
        own = [rng.standard_normal((H, T - n, D)).astype(np.float32) for _ in range(2)]
        data.append((np.concatenate([k0, own[0]], 1), np.concatenate([v0, own[1]], 1)))
    tables = np.concatenate([kv.build_table(x[h][:128].reshape(-1, 16, D)) for h in range(H) for x in (k0, v0 + 1)])
    kvb = kv.build_batched(kv.CODEC_RANS_HYBRID, lambda s: data[s], S, H, np.array(lens), D, tables, dev,
                           shared={s: (0, shared) for s in range(1, S)}, raw_groups={0: shared})
    dq = torch.from_numpy(q).to(dev)
    out = torch.full_like(dq, float("nan"))
    scale = D ** -0.5
    kvb.attention(dq, out, torch.tensor(pos, dtype=torch.int32, device=dev), scale, splits=splits, shared_groups=shared)
    got = out.cpu().double()
    for s in range(S):
        vis = pos[s] + 1
        k, v = (_dequant(x)[:, :vis] for x in data[s])
        qs = torch.from_numpy(q[s]).double().view(H, gqa, D)
        want = torch.matmul(torch.softmax(torch.matmul(qs, k.transpose(1, 2)) * scale, -1), v).view(H * gqa, D)
        # a weight's relative error is its score's absolute one: operands of 22 bits and float32 sums, 2^-21 of
        # sum |q k|, and about 2^-20 for exp, the weights' own parts and the merge; twice that for numerator and sum
        a = torch.matmul(qs.abs(), k.abs().transpose(1, 2)).amax().item() * scale
        bound = 2 * (2.0 ** -21 * a + 2.0 ** -20) * v.abs().amax().item()
        assert (got[s] - want).abs().amax().item() <= bound, (s, (got[s] - want).abs().amax().item(), bound)
