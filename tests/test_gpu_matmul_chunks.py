"""Pair-rANS matmul over the shapes where its launch changes form: one chunk of 4096 columns and several, a last chunk of
one stripe, a grid of less and more than a workgroup per CU (two fit one), one to four batch tiles and more than four,
general and aligned x. Oracle: float64 product of the decoded weights with x (as tests/test_gpu_matmul.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(48, 4096), (48, 4352), (33, 8192), (64, 12544), (17, 4500), (16 * 300 + 5, 320),
                                       (16 * 260, 4352)])
@pytest.mark.parametrize("batch", [1, 2, 17, 33, 64, 70])
def test_rans_matmul_chunks(rows, cols, batch):
    import torch
    from chromofold_amd import qw
    print(f"case {rows}x{cols} batch {batch}", flush=True)
    rng = np.random.default_rng(rows + cols + batch)
    h = qw.encode_int4((0.02 * rng.standard_normal((rows, cols))).astype(np.float32), qw.QW_CODEC_RANS)
    w = qw.QwMatrix(h, "cuda:0")
    wd = torch.from_numpy((h.sym.astype(np.float64) - 8) * np.repeat(h.scales.astype(np.float64), 64, 1)[:, :cols])
    x = torch.from_numpy(rng.standard_normal((batch, cols)).astype(np.float32)).to(torch.bfloat16)
    for shift in (0, 1):  # x at a 16-byte boundary, and two bytes past one
        buf = torch.zeros(batch * cols + 8, dtype=torch.bfloat16, device="cuda:0")
        xd = buf[shift:shift + batch * cols].view(batch, cols)
        xd.copy_(x)
        y = torch.full((batch, rows), float("nan"), device="cuda:0")
        w.matmul_into(xd, y)
        ref = x.double() @ wd.t()
        # exact products; fp32 sums of up to 12544 of them in ~200 partial sums: under 1e-6 of the row norm
        err = ((y.cpu().double() - ref).norm(dim=1) / ref.norm(dim=1)).max()
        assert float(err) <= 1e-6, (shift, float(err))
