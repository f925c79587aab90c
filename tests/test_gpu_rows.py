"""The matrix-core kernels over token rows: the hyper-connection mix
(hc_rows.hip) against the oracle's _gated_residual.

Row counts at the edges of the row tiles (16, 32, 64, 256) and of the dispatch
(8/9: one-row kernels to few-rows; 192/193 and 512/513: few to many).
Bars as for the few-row kernels: 2e-2 in bf16 (the oracle rounds to bf16 at
every step, as the kernels do), 1e-4 in float32 (another summation order).
"""

from __future__ import annotations

import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import inputs as gi  # noqa: E402

from oracle.config import OracleConfig  # noqa: E402
from oracle.mixing import OracleMixer  # noqa: E402

from margins import rel_err  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("dtype,hidden,rows", [(BF, 2048, r) for r in (8, 9, 15, 16, 17, 192, 193, 256, 257, 289)] +
                         [(F32, 2048, r) for r in (8, 9, 17, 33, 512, 513)] +
                         [(BF, 2560, 18), (BF, 2560, 200), (F32, 2560, 20), (F32, 2560, 530)])
def test_hyper_mix_rows_match_oracle(gpu, dtype, hidden, rows):
    qm = gpu
    tol = 2e-2 if dtype == BF else 1e-4
    for layer in (5, None):
        print(f"hc rows {dtype} hidden={hidden} rows={rows} layer={layer}", flush=True)
        prefix = "output_hc" if layer is None else f"blk.{layer}.hc_attn"
        store = gi.FakeStore(gi.hc_weights(prefix, 11 + rows, dtype, hidden=hidden, with_inject=layer is not None))
        model = qm.model.Qwen4MixModel(qm.config.MixConfig(hidden_size=hidden), store, device=DEV)
        oracle = OracleMixer(OracleConfig(hidden_size=hidden), store)
        hyper = gi.normal(gi.rng(rows), (1, rows, 4 * hidden), 1.0).to(dtype)
        want, _, want_inject = oracle._gated_residual(hyper, layer, "attn")
        mixed, _, inject = model._gated_residual(hyper.to(DEV), layer, "attn")
        torch.cuda.synchronize()
        assert rel_err(mixed, want, tol) < tol
        # every row by itself: a wrong row of a tile would hide in the whole
        d = (mixed.cpu().float() - want.float()).abs().amax(-1)
        assert float((d / want.float().abs().amax(-1)).max()) < 2 * tol
        if layer is None:
            assert inject is None
        else:
            assert rel_err(inject, want_inject, tol) < tol
