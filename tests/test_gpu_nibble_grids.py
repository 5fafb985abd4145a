"""Batches of more workgroups than one dimension of a launch holds (2^32 work-items, 2^24 workgroups of 256 threads): many
items of tens of thousands of query tokens over a single tail token, so that every output row is that token's V. On the
VALU kernel (head_dim 64) and the matrix-core kernel (128); the merge has a row per query token and head."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,items", [(64, 270), (128, 270)])
def test_more_workgroups_than_a_dimension_holds(D, items):
    import torch
    from chromofold_amd.sealkv import MsResolver
    qt = 65000
    assert items * qt > 1 << 24
    print(f"case D={D} items={items}", flush=True)
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(D)
    k, v = (torch.from_numpy(rng.standard_normal((1, 1, D)).astype(np.float32)).to(dev) for _ in range(2))
    res = MsResolver(1, 1, 1, D, 64)
    res.create(0)
    res.stage_active(0, 0, 0, k, v)
    q = torch.zeros((qt, 1, D), dtype=torch.bfloat16, device=dev)
    # two outputs: the last item's, and one that all the others write alike
    out = torch.full((2, qt, 1, D), float("nan"), dtype=torch.bfloat16, device=dev)
    res.execute([(0, 0, q, out[int(i == items - 1)], 0, 0.1, 0) for i in range(items)])
    torch.cuda.synchronize()
    want = v[0, 0].to(torch.bfloat16)
    assert bool((out == want).all())
    res.close()
