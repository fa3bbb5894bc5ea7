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
