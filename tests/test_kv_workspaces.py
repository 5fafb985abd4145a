"""Workspaces of prepared descriptors (BatchedKv.desc / attention): a descriptor keeps its workspace alive whatever other
descriptors are made after it, and runs on two streams never share one. The host side is checked here against a recorded
launch; the results of such runs on the GPU against calls in turn."""
import gc
import weakref

import numpy as np
import pytest


class _Stream:
    def __init__(self, handle):
        self.cuda_stream = handle


def _host_batch(S=64, H=8, D=128, groups=64):
    import torch
    from chromofold_amd import kv
    z = lambda *s: torch.zeros(s, dtype=torch.int32)  # noqa: E731
    b = kv.BatchedKv(kv.CODEC_INT8, S, H, D, groups, torch.zeros(64, dtype=torch.uint8), z(S, H, groups), z(S), None)
    q = torch.zeros((S, 4 * H, D))
    return kv, b, q, torch.empty_like(q), z(S)


def test_a_descriptor_keeps_its_workspace():
    """64 sequences of 8 heads at 4096 tokens (spans), then a larger cascade descriptor of the same object."""
    kv, b, q, o, pos = _host_batch()
    s = _Stream(1)
    d = b.desc(q, o, pos, 0.1, stream=s)
    assert d.workspace_bytes > 0
    held = weakref.ref(b.workspace)
    assert held().data_ptr() == d.workspace and held().numel() >= d.workspace_bytes
    big = b.desc(q, o, pos, 0.1, shared_groups=8, stream=s)
    assert big.workspace_bytes > d.workspace_bytes and big.workspace != d.workspace
    b.workspace = None
    gc.collect()
    assert held() is not None and held().data_ptr() == d.workspace
    del d
    gc.collect()
    assert held() is None, "kept by nothing but its descriptor"


def test_runs_on_two_streams_have_a_workspace_each(monkeypatch):
    """Descriptors prepared on one stream and run on two, and one descriptor run on both."""
    kv, b, q, o, pos = _host_batch()
    seen = []
    real = kv.A.lib()

    class Recorder:
        def __getattr__(self, name):
            return getattr(real, name)

        def cf_kv_paged_attention_batched_async(self, ref, stream):
            d = ref._obj
            seen.append((stream, d.workspace, d.workspace_bytes))
            return 0

    monkeypatch.setattr(kv.A, "lib", lambda: Recorder())
    s1, s2 = _Stream(1), _Stream(2)
    d1, d2 = (b.desc(q, o, pos, 0.1, stream=s1) for _ in range(2))
    assert d1.workspace != d2.workspace
    b.attention(q, o, pos, 0.1, stream=s1, desc=d1)
    b.attention(q, o, pos, 0.1, stream=s2, desc=d2)
    b.attention(q, o, pos, 0.1, stream=s2, desc=d1)
    assert seen[0] == (1, d1.workspace, d1.workspace_bytes)
    for stream, ws, nbytes in seen[1:]:
        assert stream == 2 and ws not in (d1.workspace, d2.workspace) and nbytes == d1.workspace_bytes
    d1.workspace, d1.workspace_bytes = None, 0  # a caller's own choice stands
    b.attention(q, o, pos, 0.1, stream=s2, desc=d1)
    assert seen[-1] == (2, None, 0)


@pytest.mark.gpu
def test_prepared_descriptors_on_the_gpu():
    """An early descriptor after a larger one was made and dropped and its memory handed out again, and descriptors
    prepared on one stream and run on two, equal the calls in turn bit for bit."""
    import torch
    from chromofold_amd import kv
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(11)
    H, gqa, D, lens = 4, 2, 128, [2500, 200, 900, 64] * 12
    data = [tuple(rng.standard_normal((H, T, D)).astype(np.float32) for _ in range(2)) for T in lens]
    kvb = kv.build_batched(kv.CODEC_INT8, lambda s: data[s], len(lens), H, np.array(lens), D, None, dev, encoder="device")
    pos = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
    qs = [torch.from_numpy(rng.standard_normal((len(lens), H * gqa, D)).astype(np.float32)).to(dev) for _ in range(2)]
    want, got = [torch.empty_like(q) for q in qs], [torch.empty_like(q) for q in qs]
    descs = [kvb.desc(q, o, pos, 0.1) for q, o in zip(qs, got)]
    for q, o in zip(qs, want):
        kvb.attention(q, o, pos, 0.1)
    big = kvb.desc(qs[0], got[0], pos, 0.1, splits=64)
    assert big.workspace_bytes > descs[0].workspace_bytes > 0
    del big
    fill = [torch.full((descs[0].workspace_bytes,), 7, dtype=torch.uint8, device=dev) for _ in range(8)]
    kvb.attention(qs[0], got[0], pos, 0.1, desc=descs[0])
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and all(bool((f == 7).all()) for f in fill)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(20):
        for s, q, o, d in zip(streams, qs, got, descs):
            kvb.attention(q, o, pos, 0.1, stream=s, desc=d)
    torch.cuda.synchronize()
    for o, w in zip(got, want):
        assert torch.equal(o, w)


@pytest.mark.parametrize("codec,S,groups,spans", [
    ("int8", 95, 46, False), ("int8", 95, 47, True), ("int8", 49, 46, False), ("int8", 49, 47, True),
    ("rans", 64, 30, False), ("rans", 64, 31, True), ("rans", 63, 14, False), ("rans", 63, 15, True)])
def test_which_full_grids_run_as_spans(codec, S, groups, spans):
    """Batches of 8 heads with more than 1.5 units per CU (256 CUs where no GPU says otherwise), which hold no workspace as
    one split: spans from six chain pairs per wavefront of INT8 groups; of rANS groups from two, from 64 sequences (two units
    per CU) on from four."""
    kv, b, q, o, pos = _host_batch(S=S, groups=groups)
    if codec == "rans":
        import torch
        b.codec, b.tables = kv.CODEC_RANS_HYBRID, torch.zeros(16 * kv.TABLE_BYTES, dtype=torch.uint8)
    d = b.desc(q, o, pos, 0.1, stream=_Stream(1))
    assert (d.workspace_bytes > 0) == spans
