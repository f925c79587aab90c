"""The ranking of scored rows (qm_qsa_select with a score buffer) against a
stable descending sort of the scores it returns: the same blocks in the same
order, ties to the lower index. Sizes either side of the ranking's branches
(counting to 128 blocks, 256 threads to 1024, 1024 threads beyond) and scores
that its bucket threshold cannot split: all equal, all zero, clustered in a
few ulps, one row of infinities."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SEQ = 3


@pytest.mark.parametrize("blocks", [34, 128, 130, 300, 1024, 1025, 3000])
@pytest.mark.parametrize("kind", ["normal", "equal", "zero", "clustered", "infinite", "outlier"])
def test_ranking_of_scored_rows(gpu, blocks, kind):
    qm = gpu
    ratio, topk = 64, 32
    print(f"rank {blocks} blocks, {kind}", flush=True)
    g = qm.native.QsaGeom(1, 16, 2, 256, 64, 4, 128, ratio, topk * ratio, 64, blocks, blocks * ratio, blocks, 1,
                          1e-6)
    gen = torch.Generator(device=DEV).manual_seed(blocks)
    iq = torch.randn(1, SEQ, 4, 128, generator=gen, device=DEV)
    bk = torch.randn(1, blocks, 128, generator=gen, device=DEV)
    if kind == "equal":
        bk[:] = bk[:, :1]
    elif kind == "zero":
        iq, bk = iq.abs(), -bk.abs()
    elif kind == "clustered":
        bk = bk[:, :1] * (1 + 1e-7 * torch.randint(0, 4, (1, blocks, 1), generator=gen, device=DEV))
    elif kind == "infinite":
        bk[:, 5:70] = 3e38
        iq = iq.abs() + 1
    elif kind == "outlier":
        bk[:, blocks // 2] *= 1e6
    # the last row sees every block, the others all but the last
    pos = torch.tensor([blocks * ratio - SEQ], dtype=torch.int32, device=DEV)
    ids = torch.full((1, SEQ, topk), -1, dtype=torch.int32, device=DEV)
    n_sel = torch.zeros(1, SEQ, dtype=torch.int32, device=DEV)
    scores = torch.empty(1, SEQ, blocks, device=DEV)
    qm.native.call("qm_qsa_select", ctypes.byref(g), SEQ, iq.data_ptr(), bk.data_ptr(), pos.data_ptr(), None,
                   ids.data_ptr(), n_sel.data_ptr(), None, scores.data_ptr(), qm.native.stream_handle())
    torch.cuda.synchronize()
    assert n_sel.tolist() == [[topk] * SEQ]
    want = torch.sort(scores.cpu(), dim=-1, descending=True, stable=True).indices[..., :topk]
    assert torch.equal(ids.cpu().long(), want)
