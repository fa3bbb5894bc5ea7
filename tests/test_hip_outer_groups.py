"""Outer products computed by the elementwise group that reads them: the same values bit for bit as
the product's own kernel followed by the group's."""
import numpy as np
import pytest

import rustautograd_amd as rg

pytestmark = pytest.mark.gpu


def _t(gen, *shape):
    return rg.tensor(gen.normal(size=shape).astype(np.float32))


def _absorbed(compiled):
    plan = compiled.plan_summary()
    return [k for k, r in enumerate(compiled._n.step_runs_in()) if r != k and plan[r]["kind"] == "fused" and plan[k].get("op", "").startswith("matmul")]


def _both(monkeypatch, fn, args):
    """The number of products inside groups, with the results equal to the separate kernels'."""
    monkeypatch.setenv("RG_HIP_PAIR", "0")
    apart = rg.compile(fn, args, device="hip", validate="none")
    monkeypatch.delenv("RG_HIP_PAIR")
    fused = rg.compile(fn, args, device="hip", validate="none")
    assert _absorbed(apart) == []
    for _ in range(3):
        for a, b in zip(apart(*args), fused(*args)):
            assert np.array_equal(np.asarray(a.numpy()).view(np.uint32), np.asarray(b.numpy()).view(np.uint32))
    return len(_absorbed(fused))


# Rows below, at and beside a block's 32 and a pass's 2, columns within, at and past a block's 256, every K edge.
@pytest.mark.parametrize("m,n,k", [(1025, 260, 1), (1031, 512, 2), (1024, 1024, 16), (3001, 256, 7), (33, 9000, 13), (262144, 4, 5), (2, 140000, 3), (547, 2052, 8)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True)])
def test_one_product_in_an_update(monkeypatch, m, n, k, ta, tb):
    print(f"{m} x {n}, K = {k}, ta {ta}, tb {tb}", flush=True)
    gen = np.random.default_rng(m + n + k)
    x, y = _t(gen, *((k, m) if ta else (m, k))), _t(gen, *((n, k) if tb else (k, n)))
    w, row = _t(gen, m, n), _t(gen, n)

    def fn(w, x, y, row):
        g = (rg.swapaxes(x, 0, 1) if ta else x) @ (rg.swapaxes(y, 0, 1) if tb else y)
        return w - 0.1 * g * row, rg.tanh(w + g)

    assert _both(monkeypatch, fn, (w, x, y, row)) == 1


def test_several_products_and_a_state_updated_in_place(monkeypatch):
    """Two layers' gradients in one group; three of K = 16, of which two fit its registers; and a
    group writing over the large product that it reads beside the outer one."""
    gen = np.random.default_rng(3)
    a, b, x, y = _t(gen, 16, 1100), _t(gen, 16, 600), _t(gen, 1100, 9), _t(gen, 9, 600)
    w, v = _t(gen, 1100, 600), _t(gen, 1100, 600)
    assert _both(monkeypatch, lambda w, v, a, b, x, y: (w - 0.5 * (rg.swapaxes(a, 0, 1) @ b), v - 0.5 * (x @ y)), (w, v, a, b, x, y)) == 2
    c = _t(gen, 1100, 16)
    assert _both(monkeypatch, lambda w, a, b, c: (w * (rg.swapaxes(a, 0, 1) @ b) + (c @ b) * ((c + 1.0) @ (b * 2.0)),), (w, a, b, c)) == 2
    p, q = _t(gen, 1100, 64), _t(gen, 64, 600)
    assert _both(monkeypatch, lambda p, q, x, y: (rg.tanh(p @ q) - x @ y,), (p, q, x, y)) == 1


def test_products_that_others_read_or_rows_not_of_four_stay_apart(monkeypatch):
    gen = np.random.default_rng(4)
    x, y, w = _t(gen, 1100, 9), _t(gen, 9, 600), _t(gen, 1100, 600)
    assert _both(monkeypatch, lambda w, x, y: (w - x @ y, x @ y), (w, x, y)) == 0
    assert _both(monkeypatch, lambda w, x, y: (w - x @ y, (x @ y).sum()), (w, x, y)) == 0
    y, w = _t(gen, 9, 602), _t(gen, 1100, 602)
    assert _both(monkeypatch, lambda w, x, y: (w - x @ y,), (w, x, y)) == 0
