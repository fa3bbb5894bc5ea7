"""Products too small to fill the chip, launched together on 32x32 fp32 tiles (k_gemm_f32_group),
against single launches (RG_HIP_PAIR=0), bit for bit: each block runs the single launch's code."""

import numpy as np
import pytest

import rustautograd_amd as rg
from rustautograd_amd import _pytree, workloads

pytestmark = pytest.mark.gpu


def test_small_products_launched_together_match_single_launches(monkeypatch):
    """C3's layers: pairs of an input and a weight gradient, and triples with the weight gradient
    before them."""
    step, state = workloads.gpt_train_step(workloads.GPT_CONFIGS["C3"])
    print("C3: compile with and without grouped products, 1 device step", flush=True)
    monkeypatch.setenv("RG_HIP_PAIR", "0")
    single = rg.compile(step, (state,), validate="none", device="hip")
    monkeypatch.delenv("RG_HIP_PAIR")
    grouped = rg.compile(step, (state,), validate="none", device="hip")
    plan, runs_in = grouped.plan_summary(), grouped._n.step_runs_in()
    products = [k for k, p in enumerate(plan) if p.get("op", "").startswith("matmul")]
    members = [runs_in[k] for k in products if runs_in[k] != k and runs_in[k] in products]
    assert len(members) >= 8 and max(members.count(r) for r in members) == 2, members
    r0, r1 = rg.run(single, state, steps=1), rg.run(grouped, state, steps=1)
    assert np.array_equal(np.array(r0.history["aux"]).view(np.uint64), np.array(r1.history["aux"]).view(np.uint64))
    for a, b in zip(_pytree.leaves(r0.state), _pytree.leaves(r1.state)):
        assert np.array_equal(np.atleast_1d(a.numpy()).view(np.uint8), np.atleast_1d(b.numpy()).view(np.uint8))


def test_a_product_is_not_moved_past_an_epilogue_that_reads_it(monkeypatch):
    """P's kernel computes X + tanh(P), a step that stands after Y in the plan: X, which would pair
    with Y at Y's step, has to be there before P."""
    gen = np.random.default_rng(5)
    a, b, c, d, e, f = (rg.tensor(gen.normal(size=s).astype(np.float32)) for s in [(64, 4096), (64, 2048), (4096, 64), (64, 2048), (64, 4096), (64, 2048)])

    def fn(a, b, c, d, e, f):
        x, p, y = rg.swapaxes(a, 0, 1) @ b, c @ d, rg.swapaxes(e, 0, 1) @ f
        return y, x + rg.tanh(p)

    monkeypatch.setenv("RG_HIP_PAIR", "0")
    single = rg.compile(fn, (a, b, c, d, e, f), device="hip", validate="none")
    monkeypatch.delenv("RG_HIP_PAIR")
    grouped = rg.compile(fn, (a, b, c, d, e, f), device="hip", validate="none")
    assert grouped._n.step_runs_in() == [0, 1, 2, 1]
    for u, v in zip(single(a, b, c, d, e, f), grouped(a, b, c, d, e, f)):
        assert np.array_equal(np.asarray(u.numpy()).view(np.uint32), np.asarray(v.numpy()).view(np.uint32))
