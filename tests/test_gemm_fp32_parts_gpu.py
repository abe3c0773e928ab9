"""fp32 GEMMs run on the bf16 matrix cores with every operand in three bf16
parts: against float64 at the edges of the tiles, and for operands that the
parts do not serve (infinities, NaN, values next to the ends of the range),
which must come out as the fp32 MFMA has them.

Tolerance: a K-long sum rounds at most 6 times per 16 of K, each time by 2^-24
of the running sum at most; with K <= 4096 normal products the measured error
is below 1e-6, the bar 2e-6."""
import numpy as np
import pytest

from oracle import reference as ora
from tests.helpers import download, normal, upload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    from qutai_amd.backends import amd

    amd.get_runtime()
    return amd


def product(amd, a, b, ta=False, tb=False, **kw):
    m, k, n = a.shape[0], a.shape[1], b.shape[1]
    left, right = upload((a.T if ta else a).ravel(), "float32"), upload((b.T if tb else b).ravel(), "float32")
    return download(amd.gemm(left, right, m, k, n, transpose_left=ta, transpose_right=tb, **kw)).reshape(m, n)


@pytest.mark.parametrize("m,k,n", [(1, 16, 1), (33, 17, 65), (128, 256, 64), (257, 130, 255), (64, 4096, 64),
                                   (520, 1000, 700), (1100, 96, 1030)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("scale", [1.0, 1e-30])
def test_against_float64(amd, m, k, n, ta, tb, scale):
    a, b = normal(m, (m, k), scale), normal(n, (k, n))
    exact = a.astype(np.float64) @ b.astype(np.float64)
    assert ora.rel_frobenius(product(amd, a, b, ta, tb), exact) <= 2e-6


def test_subnormal_operands_keep_their_bits(amd):
    a, b = normal(1, (96, 200), 3e-39), normal(2, (200, 160), 1e5)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    assert ora.rel_frobenius(product(amd, a, b), exact) <= 2e-6


# Each product of two values takes three bf16 parts of each: all of them count,
# whatever the two magnitudes are, and the sum rounds as fp32 sums do.  Where
# outputs are subnormal they round to 2^-149, whose share of the smallest rms
# here (1e-38 sqrt(40)) is below 1e-7.
@pytest.mark.parametrize("small,large", [(1e-41, 1e35), (1e-41, 1e3), (3e-39, 1e20), (3e-39, 1e5), (1e-36, 1.0),
                                         (1e-33, 1e30), (1e-20, 1e-18), (1e-30, 1e30), (1e25, 1e11), (1e-45, 1e24)])
@pytest.mark.parametrize("m,k,n", [(96, 40, 160), (300, 500, 280)])
def test_far_apart_magnitudes(amd, m, k, n, small, large):
    a, b = normal(m, (m, k), small), normal(n, (k, n), large)
    a[5] = 0  # a row of zeros stays one
    exact = a.astype(np.float64) @ b.astype(np.float64)
    for left, right, expected in ((a, b, exact), (b.T.copy(), a.T.copy(), exact.T)):
        got = product(amd, left, right)
        assert ora.rel_frobenius(got, expected) <= 2e-6
    assert not product(amd, a, b)[5].any()


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
def test_one_and_two_products_round_as_fp32_does(amd, ta, tb):
    """K = 1: the rounded product itself.  K = 2: at most one rounding of each
    product and one of their sum, half a step (2^-24 of the value) each."""
    a, b = normal(8, (300, 1)), normal(9, (1, 260))
    assert np.array_equal(product(amd, a, b, ta, tb), a * b)
    a, b = normal(10, (300, 2)), normal(11, (2, 260))
    first, second = (a[:, i:i + 1].astype(np.float64) * b[i:i + 1] for i in (0, 1))
    bound = 2.0 ** -24 * (np.abs(first) + np.abs(second) + np.abs(first + second)) * (1 + 2.0 ** -23)
    assert np.all(np.abs(product(amd, a, b, ta, tb) - (first + second)) <= bound)


@pytest.mark.parametrize("k", [3, 4, 7, 8, 15, 16])
def test_short_sums_are_as_good_as_rounded_ones(amd, k):
    """One chain of 16 of K, cut off, and one rounding (2^-24 / sqrt 3 = 3.4e-8 of
    a value in the rms): measured 3.1e-8 to 3.4e-8, where fp32 products and sums
    rounded one by one give 3.5e-8 to 7.4e-8."""
    a, b = normal(12, (500, k)), normal(13, (k, 700))
    assert ora.rel_frobenius(product(amd, a, b), a.astype(np.float64) @ b.astype(np.float64)) <= 3.6e-8


def test_infinities_nan_and_the_top_of_the_range(amd):
    a, b = normal(3, (300, 64)), normal(4, (64, 300))
    a[5, 7], a[9, 3], b[11, 13] = np.inf, np.nan, -np.inf
    a[20] = 0
    a[20, 0], b[0, 40] = 3.4e38, 0.5  # finite: next to the largest float, halved
    with np.errstate(invalid="ignore"):
        exact = a.astype(np.float64) @ b.astype(np.float64)
    got = product(amd, a, b)
    assert np.array_equal(np.isnan(got), np.isnan(exact))
    top = float(np.finfo(np.float32).max) * (1 + 2.0 ** -25)  # beyond it fp32 rounds to infinity
    assert np.array_equal(np.isposinf(got), exact > top) and np.array_equal(np.isneginf(got), exact < -top)
    finite = np.isfinite(got)
    assert ora.rel_frobenius(got[finite], exact[finite]) <= 2e-6
    assert abs(got[20, 40] / exact[20, 40] - 1) <= 2e-6
