"""Products off the large fp32 tiles: float64 on fp64 MFMA tiles, the streaming kernels at sizes no
vector divides, 16- to 31-wide outputs on matrix cores, and the wave-per-output kernel.

Bounds: a sum of K products in any order, each rounded, is within K + 1 roundings of the sum of the
magnitudes: (K + 1) 2^-53 of it in float64 and (K + 1) 2^-24 in float32, against sums in extended
precision (float64) or float64 (float32).
"""

import numpy as np
import pytest

import rustautograd_amd as rg

pytestmark = pytest.mark.gpu
FLAGS = [(False, False), (True, False), (False, True), (True, True)]


def _check(m, n, k, ta, tb, dtype, batch=()):
    gen = np.random.default_rng([m, n, k])
    a = gen.standard_normal(batch + ((k, m) if ta else (m, k))).astype(dtype)
    b = gen.standard_normal(batch + ((n, k) if tb else (k, n))).astype(dtype)

    def f(a, b):
        return (rg.swapaxes(a, -1, -2) if ta else a) @ (rg.swapaxes(b, -1, -2) if tb else b)

    print(f"{dtype} product {batch} {m} x {n} x {k}, ta {ta}, tb {tb}", flush=True)
    x, y = rg.tensor(a), rg.tensor(b)
    got = rg.compile(f, (x, y), validate="none", device="hip")(x, y).numpy()
    wide = np.longdouble if dtype == "float64" else np.float64
    x, y = ((np.swapaxes(v, -1, -2) if t else v).astype(wide) for v, t in ((a, ta), (b, tb)))
    unit = wide(2.0) ** (-53 if dtype == "float64" else -24)
    assert got.shape == batch + (m, n)
    assert np.all(np.abs(got - x @ y) <= (k + 1) * unit * (np.abs(x) @ np.abs(y)))


@pytest.mark.parametrize("m,n,k", [
    (16, 16, 4), (17, 19, 5), (31, 33, 65), (48, 700, 17),   # 16x16 tiles, the waves sharing K
    (512, 520, 40), (500, 515, 33),                          # 32x32 tiles
    (1600, 1024, 20), (1601, 1030, 17),                      # 64x64 tiles
    (1, 1, 7), (3, 5, 1000), (15, 40, 33), (2000, 1, 60), (20, 3, 5000), (300, 300, 3),   # without matrix cores
])
@pytest.mark.parametrize("ta,tb", FLAGS)
def test_float64_products(m, n, k, ta, tb):
    _check(m, n, k, ta, tb, "float64")


@pytest.mark.parametrize("m,n,k", [(20, 33, 18), (70, 70, 70), (5, 6, 40)])
def test_batched_float64_products(m, n, k):
    _check(m, n, k, False, True, "float64", (3, 5))


@pytest.mark.parametrize("m,n,k", [
    (8, 1, 256), (256, 1, 8), (1000, 1, 500), (500, 1, 400), (20000, 1, 40), (7, 9, 300), (3, 3, 31), (130, 126, 33),   # a wave per output
    (24, 200, 200), (200, 24, 200), (16, 16, 1100), (17, 500, 100),                       # 16 to 31 wide
    (4, 1609, 1609), (13, 1001, 777), (8, 67, 600), (1, 1025, 515), (1603, 1, 1603), (65, 1, 513),   # streamed: rows and dots
    (1001, 1003, 5), (130, 127, 16), (4097, 5, 3), (300, 1027, 1),                        # streamed: outer products
])
@pytest.mark.parametrize("ta,tb", FLAGS)
def test_float32_products_of_odd_sizes(m, n, k, ta, tb):
    _check(m, n, k, ta, tb, "float32")


@pytest.mark.parametrize("m,n,k", [(40, 24, 40), (33, 16, 50), (24, 24, 24), (5, 7, 60)])
def test_batched_float32_products_of_odd_sizes(m, n, k):
    _check(m, n, k, False, False, "float32", (4, 6))


def test_many_small_float64_products():
    """Sides under a 64x64 and a 32x32 tile, in batches that would fill the chip with such tiles."""
    _check(20, 20, 8, False, True, "float64", (2048,))
    _check(16, 40, 9, False, False, "float64", (1024,))


def test_the_tallest_matrix_against_a_vector():
    """2^26 - 1 rows of 32, just under the largest buffer: a wave per output would be a launch of 2^32
    threads, one more than there may be. Every value is checked on a sample of rows and at both ends."""
    rows, k = 2 ** 26 - 1, 32
    gen = np.random.default_rng(1)
    x, y, z = gen.standard_normal((rows, 1), dtype=np.float32), gen.standard_normal((1, k), dtype=np.float32), gen.standard_normal((k, 1), dtype=np.float32)
    print(f"{rows} x 1 x {k}", flush=True)
    args = tuple(rg.tensor(v) for v in (x, y, z))
    got = rg.compile(lambda x, y, z: rg.maximum(x, y) @ z, args, validate="none", device="hip")(*args).numpy()
    at = np.r_[0:1000, rows - 1000:rows, gen.integers(0, rows, 100000)]
    a = np.maximum(x[at], y).astype(np.float64)
    assert got.shape == (rows, 1)
    assert np.all(np.abs(got[at] - a @ z) <= (k + 1) * 2.0 ** -24 * (np.abs(a) @ np.abs(z)))
