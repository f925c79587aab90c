"""Prefill chunks whose rows go through the chunk attention in parts (more than
280 MB of partial outputs: 1024 rows of one sequence, 512 of two), against the
same tokens in chunks of 300 rows, which are one part and which test_gpu_qsa.py
compares with the oracle."""

from __future__ import annotations

import ctypes
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import inputs as gi  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F32 = torch.bfloat16, torch.float32
LAYER = 3
WIDTHS = (16 * 512, 512, 512, 512, 128)


def _setup(qm, dtype, batch, seed):
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.qsa_weights(LAYER, 90, dtype)), device=DEV, max_ctx=4096)
    cache = qm.MixHybridCache(LAYER + 1, model.config, batch, 4096, DEV, dtype, page_table="random", seed=3)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return model, cache, lambda n: [torch.randn(batch, n, w, generator=gen, device=DEV).to(dtype) for w in WIDTHS]


@pytest.mark.parametrize("dtype,batch,seq", [(BF, 1, 1024), (BF, 1, 1025), (BF, 1, 1333), (BF, 1, 2172), (F32, 1, 1333),
                                             (BF, 2, 700), (F32, 2, 530), (BF, 9, 260)])
def test_parts_equal_shorter_chunks(gpu, dtype, batch, seq):
    """Row by row: a wrong row of a part would hide in the whole. A row's partials
    and selection do not depend on the rows beside it, so bf16 differs by at most
    one rounding (2^-8) and float32 by the merge's order (1e-6)."""
    qm = gpu
    pos = 1500                                       # the selection is on from token 2112
    print(f"chunk of {seq} rows in parts, batch {batch} {dtype}", flush=True)
    outs, caches = [], []
    for step in (seq, 300):
        model, cache, rand = _setup(qm, dtype, batch, 6)
        model.qsa_core(*rand(pos), LAYER, cache, 0)
        x = rand(seq)
        outs.append(torch.cat([model.qsa_core(*(t[:, r:r + step].contiguous() for t in x), LAYER, cache, pos + r)
                               for r in range(0, seq, step)], 1).float())
        caches.append(cache[LAYER])
    torch.cuda.synchronize()
    err = (outs[0] - outs[1]).abs().amax(-1) / outs[1].abs().amax(-1)
    assert float(err.max()) <= (2 ** -8 if dtype == BF else 1e-6)
    assert torch.equal(caches[0].k_pool, caches[1].k_pool) and torch.equal(caches[0].block_keys, caches[1].block_keys)


@pytest.mark.parametrize("dtype,at", [(BF, 0.5), (F32, 0.5), (F32, 0.0)])
def test_outputs_over_the_queries(gpu, dtype, at):
    """qm_qsa_attend_chunk with out over the prepared queries, from ``at`` of them
    on: a part's outputs must not be stored before the next part has read its
    queries. The bits of the same call with an output of its own."""
    qm = gpu
    seq, pos = 1300, 2048
    print(f"chunk attention over q {dtype} at {at}", flush=True)
    model, cache, rand = _setup(qm, dtype, 1, 8)
    model.qsa_core(*rand(pos), LAYER, cache, 0)
    x = rand(seq)
    want = model.qsa_core(*x, LAYER, cache, pos)
    lc = cache[LAYER]
    g = model.qsa_geom(cache, dtype)
    n_ws = qm.native.load().qm_qsa_attend_chunk_workspace(ctypes.byref(g), seq)
    ws = torch.empty(n_ws, dtype=torch.uint8, device=DEV)
    q_bytes, out_bytes = lc.last_q.numel() * 2, want.numel() * want.element_size()
    start = int(q_bytes * at)
    buf = torch.empty(max(q_bytes, start + out_bytes), dtype=torch.uint8, device=DEV)
    q = buf[:q_bytes].view(BF)
    q.copy_(lc.last_q.flatten())
    out = buf[start:start + out_bytes].view(dtype)
    positions = torch.tensor([pos], dtype=torch.int32, device=DEV)
    qm.native.call("qm_qsa_attend_chunk", ctypes.byref(g), seq, q.data_ptr(), x[0].data_ptr(), lc.k_pool.data_ptr(),
                   lc.v_pool.data_ptr(), positions.data_ptr(), lc.page_table.data_ptr(), lc.last_ids.data_ptr(),
                   lc.last_n_sel.data_ptr(), out.data_ptr(), ws.data_ptr(), n_ws, qm.native.stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(out, want.flatten())
