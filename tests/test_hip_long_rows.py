"""Row groups over rows longer than a wavefront's 1024 elements (a block per row), against float64."""
import numpy as np
import pytest

import rustautograd_amd as rg
from rustautograd_amd import nn

pytestmark = pytest.mark.gpu

# Beside and at a wave's share, odd, of two and of four elements, the longest; few rows and many.
SIZES = [(5, 1025), (300, 1026), (3, 2047), (64, 2048), (257, 5000), (2, 6148), (33, 8191), (40, 8192)]


def _row_steps(c):
    return [s for s in c.plan_summary() if s["kind"] == "fused" and s["row_len"]]


def _close(got, want, dtype, length):
    """Exponentials and divisions cost a few roundings a value; a sum of `length` values at most its
    depth in roundings of its terms' sum (16 in a lane, 6 and 3 levels above)."""
    eps = np.finfo(dtype).eps
    assert np.abs(np.asarray(got.numpy(), np.float64) - want).max() <= 40 * eps * max(1.0, np.abs(want).max()), length


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("rows,length", SIZES)
def test_softmax_and_its_gradient(rows, length, dtype):
    print(rows, length, dtype, flush=True)
    gen = np.random.default_rng(length)
    xv, wv, bv = gen.normal(size=(rows, length)) * 3, gen.normal(size=(rows, length)), gen.normal(size=length)
    x, w, b = (rg.tensor(v.astype(dtype)) for v in (xv, wv, bv))
    fn = rg.value_and_grad(lambda x, w, b: (nn.softmax(x + b) * w).sum())
    c = rg.compile(lambda x, w, b: (nn.softmax(x + b), fn(x, w, b)[1]), (x, w, b), device="hip", validate="none")
    assert _row_steps(c) and all(s["row_len"] == length for s in _row_steps(c))
    z = np.asarray(x.numpy(), np.float64) + np.asarray(b.numpy(), np.float64)
    wd = np.asarray(w.numpy(), np.float64)
    e = np.exp(z - z.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    got_p, got_g = c(x, w, b)
    # exp of a difference up to 25 has that many roundings more, relative to the value.
    _close(got_p, p, dtype, length)
    _close(got_g, p * (wd - (p * wd).sum(1, keepdims=True)), dtype, length)


@pytest.mark.parametrize("rows,length", SIZES)
def test_extremes_masks_and_values_that_are_not_finite(rows, length):
    """max and min over rows of -inf, the lowest value, inf and NaN, beside whole sums."""
    gen = np.random.default_rng(rows)
    xv = gen.integers(-8, 9, size=(rows, length)).astype(np.float32)
    xv[0, -1] = np.inf
    xv[1, 7] = -np.inf
    xv[-1] = np.finfo(np.float32).min
    x = rg.tensor(xv)

    def fn(x):
        hi, lo = rg.max(x, axis=-1, keepdims=True), rg.min(x, axis=-1, keepdims=True)
        return hi, lo, rg.where(x >= hi, 1.0, 0.0), (x * 0.5 + lo).sum(axis=-1, keepdims=True)

    c = rg.compile(fn, (x,), device="hip", validate="none")
    assert _row_steps(c)
    hi, lo, at, total = (np.asarray(t.numpy()) for t in c(x))
    assert np.array_equal(hi, xv.max(1, keepdims=True)) and np.array_equal(lo, xv.min(1, keepdims=True))
    assert np.array_equal(at, (xv >= xv.max(1, keepdims=True)).astype(np.float32))
    fine = slice(2, rows - 1)
    assert np.array_equal(total[fine], (xv.astype(np.float64) * 0.5 + lo).sum(1, keepdims=True)[fine])
    assert total[0, 0] == np.inf and total[1, 0] == -np.inf and total[-1, 0] == -np.inf
    xv[2 % rows, 3] = np.nan
    y = rg.tensor(xv)
    assert np.isnan(np.asarray(c(y)[3].numpy())[2 % rows, 0])


def test_loss_over_long_rows_writes_over_what_it_reads():
    """Cross entropy of a product over 5000 classes, its gradient in the product's place, several steps."""
    gen = np.random.default_rng(9)
    xv, wv, yv = gen.normal(size=(96, 24)), gen.normal(size=(24, 5000)) * 0.2, gen.integers(0, 5000, 96)
    x, y = rg.tensor(xv.astype(np.float32)), rg.tensor(yv.astype(np.int32))

    def step(w):
        value, g = rg.value_and_grad(lambda w: nn.cross_entropy(x @ w, y))(w)
        return w - 0.5 * g, value

    w = rg.tensor(wv.astype(np.float32))
    r = rg.run(rg.compile(step, (w,), device="hip", validate="none"), w, steps=3)
    wd = np.asarray(w.numpy(), np.float64)
    for _ in range(3):
        z = np.asarray(x.numpy(), np.float64) @ wd
        p = np.exp(z - z.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        p[np.arange(96), yv] -= 1
        wd = wd - 0.5 * np.asarray(x.numpy(), np.float64).T @ p / 96
    assert np.abs(np.asarray(r.state.numpy()) - wd).max() <= 3 * 8 * np.finfo(np.float32).eps * np.abs(wd).max()
