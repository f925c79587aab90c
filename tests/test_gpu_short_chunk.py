"""Prefill chunks of 1 to 16 tokens (the token loop that forms the conv and the
gates itself, the ring written by the norm's launch) against the same tokens in
a 17-token chunk, whose conv and gates are launches of their own (checked
against the oracle elsewhere). The first part's outputs, then the rest of the 17
tokens from the state and ring that it left: a token's arithmetic is the same in
both, so float32 agrees within 1e-6 of the largest value and bf16 within one
rounding (2^-8); the rings hold inputs, unrounded, and are equal."""

from __future__ import annotations

import ctypes
from importlib import import_module

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kernel,hk,hv,seq", [(4, 16, 32, 1), (4, 16, 32, 5), (4, 2, 6, 16), (2, 3, 3, 15), (8, 1, 2, 3),
                                              (8, 2, 4, 16), (3, 2, 2, 2), (5, 1, 5, 9), (6, 1, 1, 4), (7, 1, 1, 14)])
def test_short_chunk_equals_its_tokens_in_a_longer_one(gpu, dtype, kernel, hk, hv, seq):
    native = import_module(gpu.__name__ + ".native")
    print(f"short chunk {dtype} kernel={kernel} heads={hk}/{hv} seq={seq}", flush=True)
    batch, total = 2, 17
    conv_dim = (2 * hk + hv) * 128
    gen = torch.Generator(device=DEV).manual_seed(seq * 8 + kernel)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    qkv, z = r(batch, total, conv_dim).to(dtype), r(batch, total, hv * 128).to(dtype)
    a, b = r(batch, total, hv).to(dtype), r(batch, total, hv).to(dtype)
    a_neg, dt_bias, norm_w = -r(hv).abs(), r(hv), r(128)
    conv_w = r(conv_dim, kernel).to(dtype)
    ring0, state0 = r(batch, conv_dim, kernel).to(dtype), r(batch, hv, 128, 128) * 0.1
    pos0 = torch.tensor([0, 1003], dtype=torch.int32, device=DEV)
    geom = native.DnGeom(batch, hv, hk, 128, kernel, native.act_code(dtype), 1e-6)
    lib = native.load()

    def run(t0, t1, ring, state):
        n = t1 - t0
        x = [t[:, t0:t1].contiguous() for t in (qkv, z, a, b)]
        pos = pos0 + t0
        out = torch.empty(batch, n, hv * 128, dtype=dtype, device=DEV)
        ws = torch.empty(lib.qm_dn_prefill_workspace(ctypes.byref(geom), n), dtype=torch.uint8, device=DEV)
        native.call("qm_dn_prefill", ctypes.byref(geom), n, *(native.ptr(t) for t in x), native.ptr(a_neg),
                    native.ptr(dt_bias), native.ptr(conv_w), native.ptr(norm_w), native.ptr(pos), native.ptr(ring),
                    native.ptr(state), native.ptr(out), native.ptr(ws), ws.numel(), native.stream_handle())
        torch.cuda.synchronize()
        return out.float()

    rings, states = [ring0.clone(), ring0.clone()], [state0.clone(), state0.clone()]
    want = run(0, total, rings[0], states[0])
    got = torch.cat([run(0, seq, rings[1], states[1]), run(seq, total, rings[1], states[1])], 1)
    bar = 1e-6 if dtype == torch.float32 else 2 ** -8
    err = (got - want).abs().amax((0, 2)) / want.abs().amax((0, 2))
    assert float(err.max()) <= bar, err
    assert float((states[1] - states[0]).abs().max() / states[0].abs().max()) <= 1e-6
    # outputs over the inputs' memory (not the short form): the same
    def over():
        x = [t[:, :seq].contiguous() for t in (qkv, z, a, b)]
        ring, state = ring0.clone(), state0.clone()
        ws = torch.empty(lib.qm_dn_prefill_workspace(ctypes.byref(geom), seq), dtype=torch.uint8, device=DEV)
        native.call("qm_dn_prefill", ctypes.byref(geom), seq, *(native.ptr(t) for t in x), native.ptr(a_neg),
                    native.ptr(dt_bias), native.ptr(conv_w), native.ptr(norm_w), native.ptr(pos0), native.ptr(ring),
                    native.ptr(state), native.ptr(x[0]), native.ptr(ws), ws.numel(), native.stream_handle())
        torch.cuda.synchronize()
        return x[0].flatten()[:batch * seq * hv * 128].view(batch, seq, -1).float()

    err = (over() - want[:, :seq]).abs().amax((0, 2)) / want[:, :seq].abs().amax((0, 2))
    assert float(err.max()) <= bar, err
    # the last K - 1 inputs' slots (the remaining slot holds what the part before left there)
    for i in range(batch):
        for t in range(total - kernel + 1, total):
            slot = (int(pos0[i]) + t) % kernel
            assert torch.equal(rings[1][i, :, slot], qkv[i, t])
            assert torch.equal(rings[0][i, :, slot], qkv[i, t])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,seq", [(2, 9), (3, 9), (2, 16), (3, 16), (2, 17), (3, 8), (16, 8), (17, 8), (16, 9), (17, 1)])
def test_batches_at_the_short_forms_lines(gpu, dtype, batch, seq):
    """Batches either side of where the short form stops (2 sequences, 16 up to 8
    tokens): each sequence's outputs, state and ring are those of a call of its
    own, which takes the short form up to 16 tokens. Bars as above."""
    native = import_module(gpu.__name__ + ".native")
    print(f"short chunk {dtype} batch={batch} seq={seq}", flush=True)
    hk, hv, kernel = 2, 4, 4
    conv_dim = (2 * hk + hv) * 128
    gen = torch.Generator(device=DEV).manual_seed(seq * 32 + batch)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    x = [r(batch, seq, n).to(dtype) for n in (conv_dim, hv * 128, hv, hv)]
    a_neg, dt_bias, norm_w, conv_w = -r(hv).abs(), r(hv), r(128), r(conv_dim, kernel).to(dtype)
    ring0, state0 = r(batch, conv_dim, kernel).to(dtype), r(batch, hv, 128, 128) * 0.1
    pos0 = torch.arange(batch, dtype=torch.int32, device=DEV) * 37

    def run(rows):
        n = len(range(batch)[rows])
        geom = native.DnGeom(n, hv, hk, 128, kernel, native.act_code(dtype), 1e-6)
        xs, ring, state, pos = [t[rows].contiguous() for t in x], ring0[rows].clone(), state0[rows].clone(), pos0[rows].clone()
        out = torch.empty(n, seq, hv * 128, dtype=dtype, device=DEV)
        ws = torch.empty(native.load().qm_dn_prefill_workspace(ctypes.byref(geom), seq), dtype=torch.uint8, device=DEV)
        native.call("qm_dn_prefill", ctypes.byref(geom), seq, *(native.ptr(t) for t in xs), native.ptr(a_neg),
                    native.ptr(dt_bias), native.ptr(conv_w), native.ptr(norm_w), native.ptr(pos), native.ptr(ring),
                    native.ptr(state), native.ptr(out), native.ptr(ws), ws.numel(), native.stream_handle())
        torch.cuda.synchronize()
        return out.float(), state, ring

    got = run(slice(0, batch))
    want = [torch.cat(t) for t in zip(*(run(slice(i, i + 1)) for i in range(batch)))]
    err = (got[0] - want[0]).abs().amax(2) / want[0].abs().amax(2)
    assert float(err.max()) <= (1e-6 if dtype == torch.float32 else 2 ** -8)
    assert float((got[1] - want[1]).abs().max() / want[1].abs().max()) <= 1e-6
    # every slot but the one that holds no past input, which only a longer chunk's ring write may touch
    for i in range(batch):
        for j in range(1, kernel):
            slot = (int(pos0[i]) + seq - j) % kernel
            assert torch.equal(got[2][i, :, slot], want[2][i, :, slot])
