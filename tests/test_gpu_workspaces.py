"""Workspaces that one model keeps and calls of different sizes share: every
output equals, bit for bit, the same call's on a workspace of its own."""

from __future__ import annotations

import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import inputs as gi  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16
LAYER = 3


def _pair(qm, max_ctx):
    """Two models of the same weights, each with a cache of the same pages."""
    out = []
    for _ in range(2):
        model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, BF)), device=DEV,
                                 max_ctx=max_ctx)
        out.append((model, qm.MixHybridCache(LAYER + 1, model.config, 1, max_ctx, DEV, BF, page_table="random",
                                             seed=2)))
    return out


def _inputs(gen, seq):
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(BF)  # noqa: E731
    return r(1, seq, 16 * 512), r(1, seq, 512), r(1, seq, 512), r(1, seq, 512), r(1, seq, 128)


def test_chunks_of_different_lengths_share_a_workspace(gpu):
    """Shorter chunks between longer ones: the table of selected slots of a
    longer chunk lay where a shorter one keeps its partial outputs, so it must
    not be taken for cleared memory. The selection is on from token 2112."""
    (shared, c0), (fresh, c1) = _pair(gpu, 4096)
    gen = torch.Generator(device=DEV).manual_seed(5)
    pos = 0
    for seq in (128, 2, 128, 124, 128, 512, 300, 512, 17, 512, 128):
        print(f"chunk of {seq} at {pos}", flush=True)
        x = _inputs(gen, seq)
        got = shared.qsa_core(*x, LAYER, c0, pos)
        fresh._ws.clear()
        want = fresh.qsa_core(*x, LAYER, c1, pos)
        torch.cuda.synchronize()
        assert torch.equal(got, want), (seq, pos)
        pos += seq


def test_decode_plans_of_different_sizes_share_a_workspace(gpu):
    """One layer's eager decode at positions whose plans have 66, 35, 66, 12 and
    66 items, on one workspace: the flags of a longer plan must not lie under a
    shorter plan's partials."""
    (shared, c0), (fresh, c1) = _pair(gpu, 4096)
    gen = torch.Generator(device=DEV).manual_seed(6)
    x = _inputs(gen, 2560)
    for model, cache in ((shared, c0), (fresh, c1)):
        model.qsa_core(*x, LAYER, cache, 0)
    for pos in (2500, 1100, 2500, 380, 2500, 1100, 2500):
        print(f"decode at {pos}", flush=True)
        x = _inputs(gen, 1)
        got = shared.qsa_core(*x, LAYER, c0, pos)
        fresh._ws.clear()
        want = fresh.qsa_core(*x, LAYER, c1, pos)
        torch.cuda.synchronize()
        assert torch.equal(got, want), pos
    shared.check_handoffs()
