"""fp32 products on the bf16 matrix cores (gemm_split.h), against 64-bit sums.

Shapes pick each of the tile's three sizes, whole and ragged: M and N that no tile divides (odd
ones too, so that rows start at any 4-byte address), K remainders and a K below one step, K split
over blocks, batches, every transposition.

Bounds. An operand's three bf16 parts are exact, and the terms left out of a product are at most
2^-24 of it. Within a step of 32 k a sum meets at most 24 roundings of 2^-24 and seven cut-off terms
of 2^-24 per eight, relative to the step's sum of magnitudes; each step's sum is then added with one
rounding, and so are K-split partials: an output is within (32 + K / 32 + 16) 2^-24 of the sum of its
products' magnitudes. Those roundings are random, so over a whole result the relative error is far
smaller: 0.7e-7 to 2.2e-7 measured on MI355X for K up to 8192, where the fp32 MFMA gives 2.4e-7 to
1.1e-6; 3e-7 is asserted.
"""

import numpy as np
import pytest

import rustautograd_amd as rg

pytestmark = pytest.mark.gpu


def _product(a, b, ta=False, tb=False):
    def f(a, b):
        x = rg.swapaxes(a, -1, -2) if ta else a
        y = rg.swapaxes(b, -1, -2) if tb else b
        return x @ y

    x, y = rg.tensor(a), rg.tensor(b)
    return rg.compile(f, (x, y), validate="none", device="hip")(x, y).numpy()


def _operands(m, n, k, ta, tb, batch=()):
    gen = np.random.default_rng([m, n, k])
    a = gen.standard_normal(batch + ((k, m) if ta else (m, k)), dtype=np.float32)
    b = gen.standard_normal(batch + ((n, k) if tb else (k, n)), dtype=np.float32) * np.float32(0.1)
    return a, b


def _wide(x, t):
    return (np.swapaxes(x, -1, -2) if t else x).astype(np.float64)


SHAPES = [
    # 64x64 tiles
    (1024, 1024, 96), (1000, 1028, 100), (1001, 1023, 33), (1088, 1100, 8), (65, 16640, 40),
    # 128x64 tiles
    (4096, 1536, 64), (4001, 1601, 77),
    # 128x128 tiles, whole K and K split
    (4096, 2048, 288), (4001, 2050, 300), (256, 1024, 4096), (301, 1101, 4100),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_split_products_match_64_bit_sums(m, n, k, ta, tb):
    print(f"split product {m} x {n} x {k}, ta {ta}, tb {tb}", flush=True)
    a, b = _operands(m, n, k, ta, tb)
    got = _product(a, b, ta, tb).astype(np.float64)
    x, y = _wide(a, ta), _wide(b, tb)
    want = x @ y
    err = np.abs(got - want)
    assert np.all(err <= (32 + k / 32 + 16) * 2.0 ** -24 * (np.abs(x) @ np.abs(y)))
    assert np.linalg.norm(got - want) <= 3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("m,n,k", [(96, 160, 24), (130, 129, 65)])
def test_batched_split_products_match_64_bit_sums(m, n, k):
    a, b = _operands(m, n, k, False, True, (6, 12))
    print(f"batched split product {a.shape} {b.shape}", flush=True)
    got = _product(a, b, False, True).astype(np.float64)
    want = _wide(a, False) @ _wide(b, True)
    assert np.linalg.norm(got - want) <= 3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 96), (4096, 2048, 288)])
def test_one_product_in_a_sum(m, n, k):
    """Sums with a single term that is not zero: the terms left out (1), the cut of the a1 b1 product to
    the sum of the small terms (2, a truncation) and the small terms' own roundings (2^-8 of as much):
    3.1 2^-24 of the product at most, and 4e-8 in the mean (3.5e-8 measured, an fp32 rounding is 2.5e-8)."""
    gen = np.random.default_rng(k)
    a, b = np.zeros((m, k), np.float32), gen.standard_normal((k, n), dtype=np.float32)
    a[np.arange(m), gen.integers(0, k, m)] = gen.standard_normal(m, dtype=np.float32)
    print(f"one product in a sum, {m} x {n} x {k}", flush=True)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err = np.abs(_product(a, b) - want)
    assert np.all(err <= 3.1 * 2.0 ** -24 * np.abs(want)) and np.linalg.norm(err) <= 4e-8 * np.linalg.norm(want)


@pytest.mark.parametrize("signs", [False, True])
@pytest.mark.parametrize("k", [64, 1000])
def test_operands_whose_left_out_terms_are_the_largest(k, signs):
    """1 + 2^-8 - 2^-17 squared: a2 b3 + a3 b2 + a3 b3 is 0.99 2^-24 of it, all one way, in every product
    (of either sign). Beside that a K step's sum meets the roundings above."""
    x = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    gen = np.random.default_rng(k)
    a, b = np.full((1024, k), x), np.full((k, 1024), x)
    if signs:
        a, b = (v * gen.choice(np.float32([-1, 1]), v.shape) for v in (a, b))
    print(f"the largest terms left out, K {k}, signs {signs}", flush=True)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err = np.abs(_product(a, b) - want)
    assert np.all(err <= (32 + k / 32 + 16) * 2.0 ** -24 * k * float(x) ** 2)
    assert np.linalg.norm(err) <= 3e-7 * np.linalg.norm(want)


def test_integers_up_to_24_bits_stay_exact():
    """Products and sums that fp32 holds exactly come out exactly: all three parts count."""
    gen = np.random.default_rng(3)
    a = gen.integers(-(2 ** 24) + 1, 2 ** 24, (1024, 1024)).astype(np.float32)
    b = np.zeros((1024, 1024), np.float32)
    b[gen.permutation(1024), np.arange(1024)] = gen.choice([-2.0, 0.5, 1.0], 1024)
    assert np.array_equal(_product(a, b), a.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("k", [128, 100])
def test_values_that_are_not_finite_spread_as_in_fp32(k):
    """Infinities, NaN and values at the end of fp32's range (which round past bf16's) give what fp32
    multiplication and addition give; every other output keeps its precision."""
    a, b = _operands(1024, 1024, k, False, False)
    big = np.float32(3.4e38)
    b[:] = np.where(b == 0, np.float32(0.1), b)
    a[3, 5], a[70, 9], a[500, 1], a[1000, 0] = np.inf, -np.inf, np.nan, big
    a[900, :] = 0
    a[900, 4], b[4, 7] = np.inf, np.float32(0)   # inf * 0
    b[11, 64] = np.inf
    print(f"non-finite operands, K {k}", flush=True)
    got = _product(a, b)
    with np.errstate(invalid="ignore", over="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        narrow = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(narrow)) and np.array_equal(got[np.isinf(got)], narrow[np.isinf(narrow)])
    fine = np.isfinite(got)
    fine[1000] = False
    assert np.linalg.norm((got - want)[fine]) <= 3e-7 * np.linalg.norm(want[fine])
    row = np.isfinite(got[1000])
    assert np.allclose(got[1000][row], want[1000][row], rtol=1e-5)


@pytest.mark.parametrize("m,n,k", [(1024, 1024, 96), (4096, 1536, 64), (4096, 2048, 288), (256, 1024, 4096)])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_outputs_beside_others_that_are_not_finite_keep_their_bits(m, n, k, ta, tb):
    """Infinities, NaN and huge values in some rows and columns change no bit of the others, on any
    tile and wherever their row lies in a wave's."""
    a, b = _operands(m, n, k, ta, tb)
    print(f"values that are not finite in {m} x {n} x {k}, ta {ta}, tb {tb}", flush=True)
    clean = _product(a, b, ta, tb)
    rows, cols = np.zeros(m, bool), np.zeros(n, bool)
    x, y = (a.T if ta else a), (b.T if tb else b)
    for at, value in [(3, np.inf), (20, np.nan), (100, np.float32(3.4e38)), (m - 1, -np.inf)]:
        x[at, at % k] = value
        rows[at] = True
    y[k - 1, 77] = np.nan
    cols[77] = True
    got = _product(a, b, ta, tb)
    keep = ~rows[:, None] & ~cols[None, :]
    assert np.array_equal(got[keep].view(np.uint32), clean[keep].view(np.uint32))
    assert np.all(~np.isfinite(got[[3, 20, m - 1]])) and np.all(np.isnan(got[:, 77]))
    other = np.arange(n) != 77
    want = x[100].astype(np.float64) @ y[:, other].astype(np.float64)
    fits = np.abs(want) < 3e38  # 3.4e38 times a value above 1 overflows
    assert np.any(fits) and np.allclose(got[100, other][fits], want[fits], rtol=1e-5)


def test_small_values_keep_their_precision():
    """Values down to 2^-100 (with factors that bring the products back into range) lose nothing."""
    a, b = _operands(1024, 1024, 256, False, False)
    a, b = a * np.float32(2.0 ** -100), b * np.float32(2.0 ** 90)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(_product(a, b) - want) <= 3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("exponent", [-108, -112, -120, -126, -133, -140, -146])
@pytest.mark.parametrize("small", ["left", "right", "both"])
def test_the_smallest_values_keep_their_precision(exponent, small):
    """Down to the denormal values next to 0, on either side, every bit an operand has counts: the
    bounds are those of ordinary operands. Both sides small: their products are denormal or near it,
    and each K step's sum and each addition may round to a multiple of 2^-149."""
    a, b = _operands(1024, 1024, 64, False, False)
    low, high = (exponent // 2, exponent - exponent // 2) if small == "both" else (exponent, 100)
    a, b = (np.ldexp(x, e).astype(np.float32) for x, e in zip((a, b), (high, low) if small == "right" else (low, high)))
    print(f"operands of 2^{exponent}, {small}", flush=True)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err = _product(a, b).astype(np.float64) - want
    floor = 4 * 2.0 ** -149 if small == "both" else 0.0
    assert np.all(np.abs(err) <= 50 * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + floor)
    assert np.linalg.norm(err) <= 3e-7 * np.linalg.norm(want) + floor * 1024


def test_an_error_has_no_direction():
    """Sums over many rows of a result do not collect a bias: their error is that of as many
    independent errors (twice allowed; the MFMA's own roundings, all one way, would give 15 times)."""
    gen = np.random.default_rng(8)
    a = gen.standard_normal((4096, 5000), dtype=np.float32)
    b = gen.standard_normal((256, 5000), dtype=np.float32) / np.float32(16)
    err = _product(a, b, False, True).astype(np.float64) - a.astype(np.float64) @ b.T.astype(np.float64)
    rms = np.sqrt(np.mean(err ** 2))
    assert np.sqrt(np.mean(err.sum(0) ** 2)) <= 2 * np.sqrt(4096) * rms
