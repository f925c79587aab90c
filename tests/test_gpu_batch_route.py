"""The route of a QSA decode batch: small batches over few blocks run in one
launch (Qwen4MixModel.fused_decode_fits), larger ones as prep + select + attend;
both give the same step, and bind() takes either."""

from __future__ import annotations

import os
import sys
from importlib import import_module

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import inputs as gi  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
LAYER = 3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch,pos,one_launch", [(5, 2500, True), (6, 2500, False), (8, 700, True), (9, 700, False),
                                                  (9, 200, False)])
def test_batch_routes_agree(gpu, dtype, batch, pos, one_launch):
    """Outputs of the two routes within the decode tests' 2e-2 of the largest
    value, the appended keys and values bit for bit."""
    qm = gpu
    plan = import_module(qm.__name__ + ".plan")
    print(f"decode batch {batch} at {pos} {dtype}", flush=True)
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, dtype)), device=DEV, max_ctx=4096)
    gen = torch.Generator(device=DEV).manual_seed(batch + pos)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(dtype)  # noqa: E731
    past = [r(batch, pos, n) for n in (16 * 512, 512, 512, 512, 128)]
    x = [r(batch, 1, n) for n in (16 * 512, 512, 512, 512, 128)]
    rows = torch.tensor([max(1, pos - 70 * i) for i in range(batch)], dtype=torch.int32)
    outs, caches = [], []
    for fused in (None, not one_launch):
        cache = qm.MixHybridCache(LAYER + 1, model.config, batch, 4096, DEV, dtype, page_table="random", seed=4)
        model.qsa_core(*past, LAYER, cache, 0)
        p = plan.QsaDecodePlan(model, cache, LAYER, pos, dtype, fused=fused)
        assert p.fused == (one_launch if fused is None else fused)
        p.positions.copy_(rows)
        if fused is None:
            p.bind(*x)(qm.native.stream_handle())
        else:
            p.run(*x)
        torch.cuda.synchronize()
        assert p.check() == []
        outs.append(p.out.float().clone())
        caches.append(cache[LAYER])
    assert float((outs[0] - outs[1]).abs().max() / outs[1].abs().max()) < 2e-2
    assert torch.equal(caches[0].k_pool, caches[1].k_pool) and torch.equal(caches[0].v_pool, caches[1].v_pool)


@pytest.mark.parametrize("batch,blocks,one_launch", [
    (1, 640, True), (1, 641, False), (2, 512, True), (2, 513, False), (3, 341, True), (3, 342, False), (4, 256, True),
    (4, 257, False), (5, 129, False), (5, 128, True), (7, 128, True), (8, 128, False), (7, 65, True), (6, 64, False),
    (5, 64, True), (8, 32, True), (9, 32, False), (8, 0, True)])
def test_route_at_its_lines(gpu, batch, blocks, one_launch):
    """Both routes of a step either side of every line of the rule, on caches of
    seeded random blocks: the same output within the decode tests' 2e-2."""
    qm = gpu
    plan = import_module(qm.__name__ + ".plan")
    print(f"route of {batch} x {blocks} blocks", flush=True)
    pos = blocks * 64 + 40
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, torch.bfloat16)), device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(batch + blocks)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)  # noqa: E731
    cache = qm.MixHybridCache(LAYER + 1, model.config, batch, 49152, DEV, page_table="random", seed=4)
    lc = cache[LAYER]
    lc.keys, lc.values, lc.indexer_keys = r(batch, 2, pos, 256), r(batch, 2, pos, 256), r(batch, pos, 128)
    lc.block_keys.copy_(torch.randn(lc.block_keys.shape, generator=gen, device=DEV))
    x = [r(batch, 1, n) for n in (16 * 512, 512, 512, 512, 128)]
    outs = []
    for fused in (None, not one_launch):
        p = plan.QsaDecodePlan(model, cache, LAYER, pos, torch.bfloat16, fused=fused)
        assert p.fused == (one_launch if fused is None else fused)
        p.positions.fill_(pos)
        p.run(*x)
        torch.cuda.synchronize()
        assert p.check() == []
        outs.append(p.out.float().clone())
    assert float((outs[0] - outs[1]).abs().max() / outs[1].abs().max()) < 2e-2


def test_bind_refuses_what_one_sequence_refuses(gpu):
    """A plan whose position alone is past the one-launch decode stays refused."""
    qm = gpu
    plan = import_module(qm.__name__ + ".plan")
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, torch.bfloat16)), device=DEV)
    cache = qm.MixHybridCache(LAYER + 1, model.config, 1, 49152, DEV)
    p = plan.QsaDecodePlan(model, cache, LAYER, 45000)
    x = [torch.zeros(1, 1, n, dtype=torch.bfloat16, device=DEV) for n in (16 * 512, 512, 512, 512, 128)]
    with pytest.raises(qm.native.QmError):
        p.bind(*x)


@pytest.mark.parametrize("batch,pos", [(2, 300), (9, 700), (9, 2500)])
def test_eager_decode_buffers_are_a_layers_own(gpu, monkeypatch, batch, pos):
    """Eager decode of two layers, by either route: no scratch buffer of one
    layer's step is the other's, so that the layers may run on two streams."""
    qm = gpu
    print(f"buffers of eager decode, batch {batch} at {pos}", flush=True)
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore({**gi.qsa_weights(3, 90, torch.bfloat16),
                                                           **gi.qsa_weights(7, 91, torch.bfloat16)}), device=DEV)
    cache = qm.MixHybridCache(8, model.config, batch, 4096, DEV)
    x = [torch.zeros(batch, 1, n, dtype=torch.bfloat16, device=DEV) for n in (16 * 512, 512, 512, 512, 128)]
    taken = {}
    inner = model._workspace

    def record(name, nbytes):
        buf = inner(name, nbytes)
        taken.setdefault(layer, set()).add(buf.data_ptr())
        return buf

    monkeypatch.setattr(model, "_workspace", record)
    for layer in (3, 7):
        cache[layer].ensure_qsa(batch, torch.bfloat16)
        model.qsa_core(*x, layer, cache, pos)
    torch.cuda.synchronize()
    assert taken[3] and taken[7] and not taken[3] & taken[7]


@pytest.mark.parametrize("batch,top,low", [(6, 2559, 2500), (9, 4095, 2113), (2, 41087, 41003), (1, 41087, 41050)])
def test_split_plan_covers_positions_below_its_largest(gpu, batch, top, low):
    """A split plan whose largest position completes a block, and so attends no
    tail, at positions that do: the same as the plan for that position. (Sized
    for its largest position alone, such a plan left out the tail, the newest
    tokens.)"""
    qm = gpu
    plan = import_module(qm.__name__ + ".plan")
    print(f"split plan for {top} at {low}, batch {batch}", flush=True)
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, torch.bfloat16)), device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(top)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)  # noqa: E731
    cache = qm.MixHybridCache(LAYER + 1, model.config, batch, 45056, DEV, page_table="random", seed=4)
    lc = cache[LAYER]
    lc.keys, lc.values, lc.indexer_keys = r(batch, 2, low, 256), r(batch, 2, low, 256), r(batch, low, 128)
    lc.block_keys.copy_(torch.randn(lc.block_keys.shape, generator=gen, device=DEV))
    x = [r(batch, 1, n) for n in (16 * 512, 512, 512, 512, 128)]
    outs = []
    for max_position in (low, top):
        p = plan.QsaDecodePlan(model, cache, LAYER, max_position, torch.bfloat16, fused=False)
        p.positions.fill_(low)
        p.run(*x)
        torch.cuda.synchronize()
        outs.append(p.out.float().clone())
    assert float((outs[1] - outs[0]).abs().max() / outs[0].abs().max()) < 2e-2


def test_split_plan_reports_a_position_beyond_it(gpu):
    """A batch past its plan's position: NaN and a fault in check(), as from a
    one-launch plan; the rows within it are served, and a later step is clean."""
    qm = gpu
    plan = import_module(qm.__name__ + ".plan")
    batch = 9
    print("split plan, a position beyond it", flush=True)
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, torch.bfloat16)), device=DEV)
    model.rope.get(4096)                     # the plan's tables cover the position all the same
    cache = qm.MixHybridCache(LAYER + 1, model.config, batch, 4096, DEV, page_table="random", seed=4)
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = [torch.randn(batch, 1, n, generator=gen, device=DEV).to(torch.bfloat16)
         for n in (16 * 512, 512, 512, 512, 128)]
    p = plan.QsaDecodePlan(model, cache, LAYER, 500, torch.bfloat16)
    assert not p.fused and p.batched
    p.positions.fill_(500)
    p.positions[3] = 900
    out = p.run(*x).float()
    assert out[3].isnan().all() and not out[[0, 1, 2, 4, 5, 6, 7, 8]].isnan().any()
    assert len(p.check()) == 1 and p.check() == []
    p.positions.fill_(500)
    assert not p.run(*x).isnan().any() and p.check() == []
