"""Column sums computed by another step's kernel, and what the slot they are written to holds until
then: between that kernel's step and the sum's own, no other step may read or write the slot, whose
earlier value may still be wanted.

The generated source of the plan (no device needed) shows whether a sum was taken into a product's
kernel: the kernel then has the partial rows `colp`. On the device the results equal those of the
plan with the sum in a kernel of its own (RG_HIP_EPILOGUE_SUMS=0), the sum to rounding and every
other output bit for bit.
"""

import numpy as np
import pytest

import rustautograd_amd as rg
from rustautograd_amd import _rg, nn
from test_abi import _kernel_source


def _program(k, between):
    """h's column sum s and a vector u (u = v m over K = k: 700 is split over blocks, 300 is not).
    With `between`, u is read for the last time after h's product and before s, which takes its slot."""
    def fn(v, m, x, w, q, z):
        u = v @ m
        h = rg.tanh(x @ rg.swapaxes(w, 0, 1)) * 0.5 + 1.0
        y = u @ q if between else u
        return h, y, h.sum(0).reshape(1, 1024) @ z

    return fn, _tensors((1, k), (k, 1024), (8192, 256), (1024, 256), (1024, 64), (1024, 96))


def _tensors(*shapes):
    gen = np.random.default_rng(7)
    return tuple(rg.tensor((gen.standard_normal(s) / np.sqrt(s[-1])).astype(np.float32)) for s in shapes)


def _attention_program(depth):
    """An attention layer's gradients and a chain of `depth` vector-matrix products beside them. The
    bias gradient of q, k and v is a column sum the attention backward can write; at depth 8 a product
    between the two reads the vector whose slot the sum takes."""
    layer, mask = nn.MultiHeadAttention(256, 8), rg.tril(256)

    def fn(w, b, wo, bo, x, t, v, m):
        u = v
        for _ in range(depth):
            u = u @ m
        u = u @ m[:, :64]
        params = {"qkv": {"w": w, "b": b}, "out": {"w": wo, "b": bo}}
        g = rg.grad(lambda p: nn.mse_loss(layer(p, x, mask), t))(params)
        return g["qkv"]["b"], g["qkv"]["w"], g["out"]["w"], g["out"]["b"], u

    return fn, _tensors((256, 768), (768,), (256, 256), (256,), (32, 256, 256), (32, 256, 256), (1, 768), (768, 768))


def _source(fn, args):
    from rustautograd_amd.tensor import Tracer, lift, tracing
    g = _rg.Graph()
    with tracing(g):
        out = fn(*[Tracer(g, g.input(list(t.shape), t.dtype, None)) for t in args])
        ids = [lift(g, leaf, "float32") for leaf in out]
    words, _ = _rg.plan_words(g, ids, "hip", "standard")
    return _kernel_source(words)


@pytest.mark.parametrize("k", [700, 300])
def test_a_sum_whose_slot_is_read_before_it_keeps_its_own_kernel(k):
    src = _source(*_program(k, True))
    assert src.count("rgg::gemm_mfma_block<") == 1 and "colp" not in src
    assert "colp[" in _source(*_program(k, False))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [700, 300])
@pytest.mark.parametrize("between", [True, False])
def test_results_match_the_sum_in_its_own_kernel(monkeypatch, k, between):
    fn, args = _program(k, between)
    print(f"column sum in a product's kernel, K = {k}, its slot read before it: {between}", flush=True)
    monkeypatch.setenv("RG_HIP_EPILOGUE_SUMS", "0")
    plain = rg.compile(fn, args, device="hip", validate="none")
    monkeypatch.delenv("RG_HIP_EPILOGUE_SUMS")
    fused = rg.compile(fn, args, device="hip", validate="none")
    for _ in range(3):
        (h0, y0, r0), (h1, y1, r1) = [[np.asarray(t.numpy()) for t in c(*args)] for c in (plain, fused)]
        assert np.array_equal(h0.view(np.uint32), h1.view(np.uint32)) and np.array_equal(y0.view(np.uint32), y1.view(np.uint32))
        # 8192 values of about 1 summed in another order, then 1024 such sums: far below 1e-5 of the
        # result, where a wrong operand is of the result's own size.
        assert np.linalg.norm(r1 - r0) <= 1e-5 * np.linalg.norm(r0)


@pytest.mark.gpu
@pytest.mark.parametrize("depth,between", [(8, True), (1, False)])
def test_attention_gradients_match_the_sum_in_its_own_kernel(monkeypatch, depth, between):
    fn, args = _attention_program(depth)
    print(f"column sum in the attention backward, its slot read before it: {between}", flush=True)
    monkeypatch.setenv("RG_HIP_EPILOGUE_SUMS", "0")
    plain = rg.compile(fn, args, device="hip", validate="none", optimize="standard")
    monkeypatch.delenv("RG_HIP_EPILOGUE_SUMS")
    fused = rg.compile(fn, args, device="hip", validate="none", optimize="standard")
    plan = fused.plan_summary()
    back = next(k for k, s in enumerate(plan) if s["kind"] == "attention" and s["backward"])
    total = next(k for k in range(back, len(plan)) if plan[k].get("op") == "sum")
    assert between == any(plan[total]["dst"] in plan[k].get("args", []) for k in range(back + 1, total)), plan[back:total + 1]
    assert fused._n.step_runs_in()[total] == (total if between else back)
    for _ in range(3):
        a, b = [[np.asarray(t.numpy()) for t in c(*args)] for c in (plain, fused)]
        for x, y in zip(a[1:], b[1:]):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
        # 8192 rows in another order. The key third's true sum is zero (softmax ignores a constant
        # per row), so it is measured against the whole.
        assert np.linalg.norm(a[0] - b[0]) <= 1e-5 * np.linalg.norm(a[0])
