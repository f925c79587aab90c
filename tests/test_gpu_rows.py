"""The matrix-core kernels over token rows: the hyper-connection mix
(hc_rows.hip) against the oracle's _gated_residual, and the projections
(gemm_rows.hip) against float64 products.

Row counts at the edges of the row tiles (16, 32, 64, 256) and of the dispatch
(8/9: one-row kernels to few-rows; 192/193 and 512/513: few to many).
Bars as for the few-row kernels: 2e-2 in bf16 (the oracle rounds to bf16 at
every step, as the kernels do), 1e-4 in float32 (another summation order).
"""

from __future__ import annotations

import ctypes
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


@pytest.mark.parametrize("dtype,hidden,rows", [(BF, 2048, 1041), (BF, 2048, 2000), (BF, 2560, 800), (F32, 2048, 1100)])
def test_hyper_mix_of_long_prompts_matches_oracle(gpu, dtype, hidden, rows):
    """Rows past one round of the many-rows kernel's row groups (1024 rows in bf16,
    768 at hidden 2560), where its waves take a second tile."""
    test_hyper_mix_rows_match_oracle(gpu, dtype, hidden, rows)


def _gemm_rows(qm, w, x, rows):
    m, k = x.shape
    outs = [torch.full((m, r), float("nan"), dtype=x.dtype, device=DEV) for r in rows]
    seg_rows = (ctypes.c_int * len(rows))(*rows)
    seg_out = (ctypes.c_void_p * len(rows))(*[o.data_ptr() for o in outs])
    qm.native.call("qm_gemm_rows", qm.native.act_code(x.dtype), m, w.shape[0], k, w.data_ptr(), x.data_ptr(),
                   len(rows), seg_rows, seg_out, qm.native.stream_handle())
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("dtype,k", [(BF, 2048), (BF, 4096), (F32, 1024), (F32, 2048), (F32, 4096)])
@pytest.mark.parametrize("m", [1, 5, 15, 16, 17, 33, 64])
def test_gemm_rows_matches_fp64_product(gpu, dtype, k, m):
    """qm_gemm_rows against a float64 product of the same operands: bf16 within
    one rounding of the result (2^-8 of its row's largest value), float32 within
    1e-5 (the sums' order). Segments: the DeltaNet layer's, a ragged split whose
    bounds and lengths are no multiples of 4, and fewer rows than a tile."""
    qm = gpu
    g = torch.Generator(device=DEV).manual_seed(m * 7 + k)
    for rows in ([8192, 4096, 32, 32], [600, 1, 398], [7]):
        n = sum(rows)
        print(f"gemm_rows {dtype} m={m} k={k} rows={rows}", flush=True)
        w = (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(dtype)
        x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
        want = x.double() @ w.double().t()
        got = torch.cat([o.double() for o in _gemm_rows(qm, w, x, rows)], 1)
        bar = 2 ** -8 if dtype == BF else 1e-5
        assert float(((got - want).abs().amax(1) / want.abs().amax(1)).max()) < bar


@pytest.mark.parametrize("dtype,k", [(BF, 4096), (F32, 2048)])
@pytest.mark.parametrize("m,streams", [(5, 4), (17, 4), (64, 1), (20, 10)])
def test_gemm_rows_reinject_equals_its_two_steps(gpu, dtype, k, m, streams):
    """qm_gemm_rows_reinject == qm_gemm_rows, then the reinjection's two
    roundings in torch, bit for bit."""
    qm = gpu
    n = 2048
    g = torch.Generator(device=DEV).manual_seed(31 * m + k + streams)
    print(f"gemm_rows_reinject {dtype} m={m} k={k} streams={streams}", flush=True)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(dtype)
    x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    hyper = torch.randn(m, streams * n, generator=g, device=DEV).to(dtype)
    inject = (2 * torch.sigmoid(torch.randn(m, streams, generator=g, device=DEV))).to(dtype)
    branch = _gemm_rows(qm, w, x, [n])[0]
    scaled = (branch.float()[:, None, :] * inject.float()[:, :, None]).to(dtype).float()
    want = (hyper.float().view(m, streams, n) + scaled).to(dtype).view(m, streams * n)
    got = hyper.clone()
    qm.native.call("qm_gemm_rows_reinject", qm.native.act_code(dtype), m, n, k, w.data_ptr(), x.data_ptr(), streams,
                   inject.data_ptr(), got.data_ptr(), qm.native.stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_project_routes_by_rows(gpu):
    """Layer projections at 5 and 64 rows (qm_gemm_rows) and at 65 (the library)
    equal F.linear; an input that is differentiated, or not 16-byte aligned,
    keeps F.linear."""
    qm = gpu
    store = gi.FakeStore(gi.dn_weights(0, 31, BF))
    model = qm.Qwen4MixModel(qm.MixConfig(), store, device=DEV, max_ctx=256)
    for seq in (5, 64, 65):
        hidden = gi.normal(gi.rng(32 + seq), (1, seq, gi.HIDDEN)).to(BF).to(DEV)
        for x in (hidden, hidden.clone().requires_grad_(),
                  torch.cat([hidden.new_zeros(1), hidden.flatten()])[1:].view_as(hidden)):
            got = model.project(x, 0, "dn_in")
            assert got[0].requires_grad == x.requires_grad
            for t, name in zip(got, model.PROJ_GROUPS["dn_in"]):
                want = torch.nn.functional.linear(hidden.float(), store.get(f"blk.0.{name}").to(DEV).float())
                assert rel_err(t.detach(), want, 1e-2) < 1e-2, (seq, name)


@pytest.mark.parametrize("dtype,rows,at", [(BF, 9, 0), (BF, 40, 3), (BF, 300, 0), (F32, 17, 1), (F32, 600, 0)])
def test_hyper_mix_into_the_residuals_memory(gpu, dtype, rows, at):
    """mixed over the memory of hyper (from its row ``at`` on): the bits of the
    same rows in calls of 8, whose kernels read hyper before anything is stored
    (the matrix-core kernels read it again beside the stores, and their sums have
    another order)."""
    qm = gpu
    print(f"hc over its input {dtype} rows={rows} at={at}", flush=True)
    store = gi.FakeStore(gi.hc_weights("output_hc", 5, dtype, hidden=2048, with_inject=False))
    model = qm.Qwen4MixModel(qm.MixConfig(), store, device=DEV)
    hyper = gi.normal(gi.rng(rows), (1, rows, 4 * 2048), 1.0).to(dtype).to(DEV)
    want = torch.cat([model._gated_residual(h, None, "attn")[0] for h in hyper.split(8, 1)], 1)
    over = hyper.flatten()[at * 4 * 2048:][:rows * 2048].view(1, rows, 2048)
    mixed, _, _ = model._gated_residual(hyper, None, "attn", mixed=over)
    torch.cuda.synchronize()
    assert mixed.data_ptr() == over.data_ptr() and torch.equal(mixed, want)


@pytest.mark.parametrize("rows", [9, 17, 193])
def test_bf16_gates_equal_the_precise_chains(gpu, rows):
    """Every bf16 value but the NaNs as the gate's input, 2048 a call: low-rank
    value 1 (silu(1.28125) rounds to it) times an up weight of that value, so the
    output is the rounded sigmoid itself. The matrix-core kernels' short form
    gives the bits of the vector kernels' precise one (8 rows)."""
    qm = gpu
    k = 4 * 2048
    values = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(BF)
    values = torch.where(values.isnan(), torch.zeros_like(values), values).to(DEV)
    norm_w = torch.ones(k, device=DEV)
    down = torch.zeros(320, k, dtype=BF, device=DEV)
    down[0, 0] = 4 * 1.28125
    hyper = torch.ones(rows, k, dtype=BF, device=DEV)
    up = torch.zeros(k, 320, dtype=BF, device=DEV)
    print(f"gates of {rows} rows", flush=True)

    def mix(n):
        g = qm.native.HcGeom(n, 4, 2048, 320, qm.native.act_code(BF), 1e-6)
        ws = torch.empty(qm.native.load().qm_hc_mix_workspace(ctypes.byref(g)), dtype=torch.uint8, device=DEV)
        out = torch.empty(n, 2048, dtype=BF, device=DEV)
        qm.native.call("qm_hc_mix", ctypes.byref(g), hyper.data_ptr(), norm_w.data_ptr(), down.data_ptr(), 0,
                       up.data_ptr(), out.data_ptr(), None, ws.data_ptr(), ws.numel(), qm.native.stream_handle())
        torch.cuda.synchronize()
        return out.view(torch.int16)

    for v in values.split(2048):
        up[:, 0] = v.repeat(4)
        want = mix(8)
        assert torch.equal(want[0].view(BF).float(), torch.sigmoid(v.float()).to(BF).float()) or v.float().amin() < -87
        assert torch.equal(mix(rows), want[:1].expand(rows, -1))


def test_project_stays_visible_to_torch(gpu, monkeypatch):
    """What intercepts, casts or records F.linear sees the projections of 5 rows
    too: autocast, dispatch and function modes, tensor subclasses, jit.trace,
    fake tensors. Without any, and with a default device, they are one launch."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    qm = gpu
    model = qm.Qwen4MixModel(qm.MixConfig(), gi.FakeStore(gi.dn_weights(0, 31, BF)), device=DEV, max_ctx=256)
    x, y = (gi.normal(gi.rng(s), (1, 5, gi.HIDDEN)).to(BF).to(DEV) for s in (1, 2))
    n = len(model.PROJ_GROUPS["dn_in"])
    inner, native_calls, seen = qm.native.call, [], []
    monkeypatch.setattr(qm.native, "call", lambda name, *a: (native_calls.append(name), inner(name, *a))[1])

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            if func is torch.nn.functional.linear:
                seen.append("linear")
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    want = model.project(x, 0, "dn_in")
    assert native_calls == ["qm_gemm_rows"]
    with torch.device(DEV):
        model.project(x, 0, "dn_in")
    assert native_calls == ["qm_gemm_rows"] * 2
    native_calls.clear()
    with torch.autocast("cuda", dtype=torch.float16):
        assert [t.dtype for t in model.project(x, 0, "dn_in")] == [torch.float16] * n
    with Dispatch():
        model.project(x, 0, "dn_in")
    assert sum("mm" in s for s in seen) == n
    seen.clear()
    with Function():
        model.project(x, 0, "dn_in")
    assert seen == ["linear"] * n
    assert all(type(t) is Sub for t in model.project(x.as_subclass(Sub), 0, "dn_in"))
    traced = torch.jit.trace(lambda t: tuple(model.project(t, 0, "dn_in")), (x,), check_trace=False)
    for a, b in zip(traced(y), model.project(y, 0, "dn_in")):
        assert rel_err(a, b, 1e-2) < 1e-2
    native_calls.clear()
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        fake = model.project(mode.from_tensor(x), 0, "dn_in")
    assert [t.shape for t in fake] == [t.shape for t in want] and not native_calls
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("rows,as_rows", [(9, 1), (14, 1), (14, 2), (33, 8), (200, 9), (530, 192), (20, 1000)])
def test_hyper_mix_as_has_the_bits_of_that_row_count(gpu, dtype, rows, as_rows):
    """qm_hc_mix_as over ``rows`` rows == qm_hc_mix over the same rows, as_rows at
    a time, mixed and inject, bit for bit."""
    qm = gpu
    print(f"mix of {rows} rows as {as_rows} {dtype}", flush=True)
    store = gi.FakeStore(gi.hc_weights("blk.5.hc_attn", 5, dtype, hidden=2048))
    model = qm.Qwen4MixModel(qm.MixConfig(), store, device=DEV)
    n = max(rows, as_rows)
    n += -n % as_rows
    hyper = gi.normal(gi.rng(rows), (1, n, 4 * 2048), 1.0).to(dtype).to(DEV)
    parts = [model._gated_residual(h, 5, "attn") for h in hyper.split(as_rows, 1)]
    mixed, _, inject = model._gated_residual(hyper[:, :rows], 5, "attn", as_rows=as_rows)
    torch.cuda.synchronize()
    assert torch.equal(mixed, torch.cat([p[0] for p in parts], 1)[:, :rows])
    assert torch.equal(inject, torch.cat([p[2] for p in parts], 1)[:, :rows])
