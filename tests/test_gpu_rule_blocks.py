"""The token-loop delta rule (dn_recurrent_kernel) at the edges of its 16-token
blocks, against the recurrence in float64 (oracle/f64.py is its CPU form; the
loop here is the same three lines). Bars: float32 outputs and state within 1e-5
of the largest value (128-term sums in another order), bf16 outputs within one
rounding (2^-8)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rule64(q, k, v, g, beta, S):
    q, k, v, g, beta, S = (t.double() for t in (q, k, v, g, beta, S))
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) / q.shape[-1] ** 0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    out = torch.empty_like(v)
    for t in range(q.shape[1]):
        S = S * g[:, t].exp()[..., None, None]
        d = (v[:, t] - (S * k[:, t][..., None]).sum(-2)) * beta[:, t][..., None]
        S = S + k[:, t][..., None] * d[..., None, :]
        out[:, t] = (S * q[:, t][..., None]).sum(-2)
    return out, S


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,heads,seq", [(1, 32, 1), (2, 3, 15), (1, 32, 16), (1, 5, 17), (3, 2, 33), (1, 32, 64)])
def test_recurrent_rule_blocks(gpu, dtype, batch, heads, seq):
    from importlib import import_module
    layers = import_module(gpu.__name__ + ".layers")
    print(f"recurrent rule {dtype} batch={batch} heads={heads} seq={seq}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(seq * 31 + heads)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    q, k, v = (r(batch, seq, heads, 128).to(dtype) for _ in range(3))
    g, beta = -r(batch, seq, heads).abs(), torch.sigmoid(r(batch, seq, heads))
    S = r(batch, heads, 128, 128) * 0.1
    want, want_S = rule64(q, k, v, g, beta, S)
    out, state = layers.recurrent_gated_delta_rule(q, k, v, g, beta, S)
    torch.cuda.synchronize()
    bar = 1e-5 if dtype == torch.float32 else 2 ** -8
    # per token: a wrong token of a block would hide in the whole
    err = (out.double() - want).abs().amax((2, 3)) / want.abs().amax((2, 3))
    assert float(err.max()) < bar
    assert float((state.double() - want_S).abs().max() / want_S.abs().max()) < 1e-5


@pytest.mark.parametrize("seq", [15, 16, 23, 24, 25])
def test_prefill_rule_at_the_dispatch(gpu, seq):
    """qm_dn_prefill either side of the lines between its forms (16 tokens: the
    loop forms the conv itself; 32: the chunked rule): the same prompt one token at a time through the
    decode path. bf16 outputs within 2e-2 of the largest value, the state within
    1e-3 (the bars of the decode and prefill tests)."""
    qm = gpu
    import os
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
    import inputs as gi
    bf = torch.bfloat16
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.dn_weights(0, 7, bf)), device=DEV, max_ctx=64)
    gen = torch.Generator(device=DEV).manual_seed(seq)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(bf)  # noqa: E731
    qkv, z, a, b = r(1, seq, 8192), r(1, seq, 4096), r(1, seq, 32), r(1, seq, 32)
    print(f"prefill rule seq={seq}", flush=True)
    one, many = (qm.MixHybridCache(1, model.config, 1, 64, DEV, bf) for _ in range(2))
    got = model.dn_core(qkv, z, a, b, 0, many[0])
    rows = [slice(t, t + 1) for t in range(seq)]
    want = torch.cat([model.dn_core(*(x[:, s].contiguous() for x in (qkv, z, a, b)), 0, one[0]) for s in rows], 1)
    torch.cuda.synchronize()
    assert float((got.float() - want.float()).abs().max() / want.float().abs().max()) < 2e-2
    assert float((many[0].recurrent_state - one[0].recurrent_state).abs().max()) < 1e-3
    assert torch.equal(many[0].conv_state, one[0].conv_state)


@pytest.mark.parametrize("seq", [17, 31, 32, 33, 34])
def test_prefill_rule_at_the_chunked_line(gpu, seq):
    test_prefill_rule_at_the_dispatch(gpu, seq)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,heads,seq", [(2, 32, 1216), (3, 24, 1000), (1, 100, 7808)])
def test_chunked_rule_in_segments(gpu, dtype, batch, heads, seq):
    """The chunked rule over more records than one segment takes, for several
    sequences and (7808 tokens of 100 heads) with a last segment of two chunks,
    whose preparation is split in four, against the token loop. Per token, of its
    largest value: the chunked form's operands have 16 bits (2^-16, summed over 64
    tokens: a few times that), and bf16 rounds both outputs, each by up to half a
    step of its 8 bits (2^-8)."""
    from importlib import import_module
    layers = import_module(gpu.__name__ + ".layers")
    print(f"segments {dtype} batch={batch} heads={heads} seq={seq}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(seq + heads)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    q, k, v = (r(batch, seq, heads, 128).to(dtype) for _ in range(3))
    g, beta = -r(batch, seq, heads).abs(), torch.sigmoid(r(batch, seq, heads))
    S = r(batch, heads, 128, 128) * 0.1
    want, want_S = layers.recurrent_gated_delta_rule(q, k, v, g, beta, S)
    out, state = layers.chunk_gated_delta_rule(q, k, v, g, beta, S)
    torch.cuda.synchronize()
    bar = 8 * 2 ** -16 + (2 * 2 ** -8 if dtype == torch.bfloat16 else 0)
    err = (out.float() - want.float()).abs().amax((2, 3)) / want.float().abs().amax((2, 3))
    print(f"  worst token {float(err.max()):.2e}", flush=True)
    assert float(err.max()) < bar
    assert float((state - want_S).abs().max() / want_S.abs().max()) < 8 * 2 ** -16


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_prefill_in_segments_equals_shorter_calls(gpu, dtype):
    """Two prompts of 1216 tokens through a DeltaNet core (16 q/k heads for 32
    value heads; two segments) == their first 640 and last 576 tokens in calls of
    one segment each, whose chunks are the same."""
    qm = gpu
    import os
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
    import inputs as gi
    seq, cut = 1216, 640
    print(f"prefill in segments {dtype}", flush=True)
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.dn_weights(0, 7, dtype)), device=DEV, max_ctx=64)
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = [torch.randn(2, seq, n, generator=gen, device=DEV).to(dtype) for n in (8192, 4096, 32, 32)]
    one, two = (qm.MixHybridCache(1, model.config, 2, 2048, DEV, dtype) for _ in range(2))
    got = model.dn_core(*x, 0, one[0])
    want = torch.cat([model.dn_core(*(t[:, s].contiguous() for t in x), 0, two[0])
                      for s in (slice(0, cut), slice(cut, seq))], 1)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert torch.equal(one[0].recurrent_state, two[0].recurrent_state)
    assert torch.equal(one[0].conv_state, two[0].conv_state)


@pytest.mark.parametrize("over", ["v", "q", "g"])
def test_chunked_rule_into_its_inputs_memory(gpu, over):
    """2304 tokens of 32 heads are more records than one segment takes (160 MB).
    Outputs whose first half lies over the second half of an input: the bits of
    the same call with outputs of their own."""
    native = gpu.native
    bf = torch.bfloat16
    heads, seq = 32, 2304
    print(f"chunked rule over {over}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(9)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    n = seq * heads * 128
    x = {i: r(1, seq, heads, 128).to(bf) for i in "qkv"}
    x["g"], x["beta"] = -r(1, seq, heads).abs(), torch.sigmoid(r(1, seq, heads))
    state0 = r(1, heads, 128, 128) * 0.1
    lib = native.load()
    ws = torch.empty(lib.qm_dn_chunked_workspace(1, seq, heads, 128), dtype=torch.uint8, device=DEV)

    def run(x, out):
        state = state0.clone()
        native.call("qm_dn_chunked", native.act_code(bf), 1, seq, heads, 128, *(x[i].data_ptr() for i in
                    ("q", "k", "v", "g", "beta")), state.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(),
                    native.stream_handle())
        torch.cuda.synchronize()
        return out.clone(), state

    want, want_state = run(x, torch.empty(n, dtype=bf, device=DEV))
    # the input at the start of a buffer, the outputs from the middle of the input on
    size = x[over].numel() * x[over].element_size()
    buf = torch.empty(size // 2 + 2 * n, dtype=torch.uint8, device=DEV)
    held = buf[:size].view(x[over].dtype).view(x[over].shape)
    held.copy_(x[over])
    got, state = run(dict(x, **{over: held}), buf[size // 2:].view(bf))
    assert torch.equal(got, want) and torch.equal(state, want_state)
