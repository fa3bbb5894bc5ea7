"""Products of at most 16 rows (or one column) over a long K: the row, dot and block-per-output kernels,
which of them a product takes, and the error of their sums against 64-bit ones.

A sum's rounding error: each addition errs by 0.42 2^-24 of its result (root mean square over
mantissas), so a sum of random terms that meets additions of f_1, f_2, ... of its terms has a
relative error of about 0.42 2^-24 sqrt(f_1 + f_2 + ...). A block per output: a lane's up to 5 terms
(3), six butterfly levels, up to 16 wave sums (8.5): sqrt(14) gives 0.95e-7 for the K here. Row kernel:
16 terms at a time (8.5), up to 5 of those (3), 4 waves (2.25), 16 splits (8.5): 1.2e-7. Dot kernel: four
terms at a time (2.5), 4 of those (2.5), six levels, up to 4 splits (2.5): 0.95e-7. 15 % more is allowed,
30 % for results of under 1000 values, whose own spread is that large. (Summed a term after the
other, the row kernel's quarters gave 1.5e-7 to 1.8e-7.)
"""

import numpy as np
import pytest

import rustautograd_amd as rg
from test_hip_small_products import _check

pytestmark = pytest.mark.gpu
TINY, ROWS, DOTS = 0.95e-7, 1.2e-7, 0.95e-7


def _product(a, b, ta, tb):
    def f(a, b):
        return (rg.swapaxes(a, 0, 1) if ta else a) @ (rg.swapaxes(b, 0, 1) if tb else b)

    x, y = rg.tensor(a), rg.tensor(b)
    return rg.compile(f, (x, y), validate="none", device="hip")(x, y).numpy()


@pytest.mark.parametrize("m,n,k,ta,tb,expected", [
    (1, 66, 513, False, False, TINY), (8, 66, 1000, False, False, TINY), (3, 515, 1000, False, False, TINY), (16, 257, 515, False, False, TINY),
    (77, 1, 4097, True, False, TINY), (1, 1001, 1000, False, True, TINY), (16, 1001, 513, False, True, TINY), (1000, 1, 513, False, False, TINY),
    (8, 1024, 4096, False, False, ROWS), (3, 1001, 4096, False, False, ROWS), (12, 515, 2050, False, False, ROWS), (16, 1001, 1000, False, False, ROWS),
    (16, 1023, 513, True, False, ROWS), (4096, 1, 4096, True, False, ROWS), (8, 2050, 2050, True, False, ROWS),
    (8, 2050, 2050, False, True, DOTS), (16, 1024, 2050, False, True, DOTS), (5, 3001, 1000, False, True, DOTS), (4096, 1, 4096, False, False, DOTS),
])
def test_errors_of_skinny_sums(m, n, k, ta, tb, expected):
    gen = np.random.default_rng([m, n, k])
    a = gen.standard_normal((k, m) if ta else (m, k), dtype=np.float32)
    b = gen.standard_normal((n, k) if tb else (k, n), dtype=np.float32)
    print(f"skinny sums {m} x {n} x {k}, ta {ta}, tb {tb}", flush=True)
    want = (a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64)
    assert np.linalg.norm(_product(a, b, ta, tb) - want) <= (1.15 if m * n >= 1000 else 1.3) * expected * np.linalg.norm(want)


# Row kernel: a wave's share of K at and around its 8, 16 and 64 k (K split by 4 waves and up to 16
# splits), and many times that; columns at and around a lane's 4 and a block's 256.
@pytest.mark.parametrize("m,n,k", [
    (8, 4096, 512), (8, 4097, 513), (7, 5000, 575), (9, 2051, 1023), (16, 2050, 1024), (15, 1030, 1025), (1, 9000, 1089), (2, 4100, 5000),
    (13, 260, 70001), (16, 65, 70000), (8, 1025, 4161), (3, 4098, 4096),
])
@pytest.mark.parametrize("ta", [False, True])
def test_row_kernel_at_its_edges(m, n, k, ta):
    _check(m, n, k, ta, False, "float32")


@pytest.mark.parametrize("ta", [False, True])
def test_infinities_in_a_row_kernel_reach_their_own_outputs_alone(ta):
    """Values past a wave's last whole eight k, and past its share, multiply nothing."""
    m, n, k = 11, 2049, 1003
    gen = np.random.default_rng(2)
    a, b = gen.standard_normal((m, k), dtype=np.float32), gen.standard_normal((k, n), dtype=np.float32)
    a[0, k - 1], a[3, 0], b[k - 1, 17], b[62, 900] = np.inf, -np.inf, np.inf, np.nan
    print(f"infinities in 11 x 2049 x 1003, ta {ta}", flush=True)
    got = _product(np.ascontiguousarray(a.T) if ta else a, b, ta, False)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
