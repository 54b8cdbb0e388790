"""fp32 products as halves, pairs times triples with a scale per row (csrc/h2.h): edges of tiles and of K splits, rows longer than what the split keeps in
registers, rows of any size, against float64.

Bound: a pair holds an element to 2^-23 of itself (to 2^-39 of its row's largest below 2^-16 of it), a triple exactly (to 2^-39 below 2^-15); what is left out of a product is below
2^-22 of |a||b|; the accumulator takes four products per 32 columns and rounds each time, 2^-24 of at most the sum of the magnitudes, twice that for what a matrix
instruction rounds inside: (2^-21 + (K / 8 + 8) 2^-23) sum |a||b|, and 2^-38 of the largest products for the small ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bound(a, b):
    a, b = np.abs(a.astype(np.float64)), np.abs(b.astype(np.float64))
    k = a.shape[1]
    return (2.0 ** -21 + (k / 8 + 8) * 2.0 ** -23) * (a @ b.T) + k * 2.0 ** -38 * np.outer(a.max(axis=1), b.max(axis=1)) + 1e-44


@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (65, 64, 32), (64, 130, 96), (129, 127, 64), (517, 768, 832), (200, 768, 2048), (1000, 2400, 768), (70, 40, 4128),
                                   (4100, 2050, 96), (150, 2048, 5888)])
def test_against_float64(pkg, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)
    r = rng.standard_normal((m, n), dtype=np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64).T
    got, _ = pkg.selftest_gemm(a, b, r, pairs=True)
    assert np.all(np.abs(got - (want + r)) <= bound(a, b) + 2.0 ** -23 * np.abs(want + r))
    if n % 2 == 0:
        g, u = want[:, 0::2], want[:, 1::2]
        silu = lambda x: x / (1.0 + np.exp(-x))
        got, _ = pkg.selftest_gemm(a, b, swiglu=True, pairs=True)
        bd = bound(a, b)
        slack = 1.1 * bd[:, 0::2] * np.abs(u) + np.abs(silu(g)) * bd[:, 1::2] + 1.1 * bd[:, 0::2] * bd[:, 1::2]  # |silu'| <= 1.1
        assert np.all(np.abs(got - silu(g) * u) <= slack + 2.0 ** -20 * np.abs(silu(g) * u))


def test_rows_of_any_size(pkg):
    """Rows of zeros, of subnormals, near the top of the range, and of elements 2^40 apart; their products with rows that bring them back."""
    rng = np.random.default_rng(9)
    m, n, k = 96, 80, 256
    a = rng.standard_normal((m, k)) * np.exp2(rng.integers(-20, 21, size=(m, k)))
    a *= np.exp2(np.linspace(-140, 100, m))[:, None]
    a[5] = 0
    b = rng.standard_normal((n, k)) * np.exp2(np.linspace(-100, 20, n))[:, None]
    b[7] = 0
    a, b = a.astype(np.float32), b.astype(np.float32)
    with np.errstate(over="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64).T
    got, _ = pkg.selftest_gemm(a, b, pairs=True)
    inside = np.abs(want) < 3.3e38
    assert inside.mean() > 0.9 and np.all(got[5] == 0) and np.all(got[:, 7] == 0)
    assert np.all(np.abs(got[inside] - want[inside]) <= bound(a, b)[inside] + 2.0 ** -149)


def test_no_further_from_float64_than_planes(pkg):
    for k in (768, 2048):
        rng = np.random.default_rng(k)
        a = rng.standard_normal((640, k), dtype=np.float32)
        b = rng.standard_normal((2048, k), dtype=np.float32) * np.float32(0.02)
        want = a.astype(np.float64) @ b.astype(np.float64).T
        err = {p: np.linalg.norm(pkg.selftest_gemm(a, b, pairs=p)[0] - want) / np.linalg.norm(want) for p in (True, False)}
        print(f"K {k}: pairs {err[True]:.2e}, planes {err[False]:.2e}")
        assert err[True] <= err[False]


def test_a_row_that_is_not_finite_spoils_that_row_alone(pkg):
    rng = np.random.default_rng(3)
    a = rng.standard_normal((100, 96), dtype=np.float32)
    b = rng.standard_normal((64, 96), dtype=np.float32)
    want, _ = pkg.selftest_gemm(a, b, pairs=True)
    a[17, 5], a[40, 0], a[99, 95] = np.inf, np.nan, -np.inf
    got, _ = pkg.selftest_gemm(a, b, pairs=True)
    bad = np.zeros(100, bool)
    bad[[17, 40, 99]] = True
    assert not np.isfinite(got[bad]).any() and np.array_equal(got[~bad], want[~bad])


@pytest.mark.parametrize("m,n,k", [(65, 64, 64), (70, 66, 192), (90, 2048, 2048), (150, 2048, 5888), (300, 200, 320)])
def test_halves_in_slices_shared_by_two_groups(pkg, m, n, k):
    """One slice (the second group has none), an odd number, K splits of unequal parts; products of halves are exact in fp32, so only the accumulation rounds."""
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float16).astype(np.float32)
    b = (rng.standard_normal((n, k)) * 0.02).astype(np.float16).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64).T
    got, _ = pkg.selftest_gemm(a, b, f16=True)
    assert np.all(np.abs(got - want) <= (k / 16 + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T))
