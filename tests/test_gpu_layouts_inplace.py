"""Large operands and results stored by coefficient go through polfirst copies
kept in the buffers of their own transforms: an operand's copy is read by the
transform that writes over it, a result's is written by the inverse transform that
reads it.  Here that meets every kind of transform: whole ones of 2^14 and 2^15
points, split ones, those of several passes (2^16 and 2^17 points), a single prime
and three; and middle products, whose small operand is reversed on the way.
Products are checked by evaluation at a random point and the stored forms against
polfirst ones; middle products against the middle of the product."""
import numpy as np
import pytest

import linbox_amd as lbx
from linbox_amd import PolynomialMatrix, PolynomialMatrixFFTMulDomain, PolynomialMatrixMulDomain
from polycheck import check_by_evaluation
from test_gpu_parity import ctx, rand, say, METHODS  # noqa: F401

pytestmark = pytest.mark.gpu

BY_COEFFICIENT = [("matfirst", "matfirst", "matfirst"), ("matrowfirst", "matfirst", "matrowfirst")]


@pytest.mark.parametrize("p,m,k,n,sa,sb", [
    (998244353, 40, 36, 33, 8000, 8100),    # 2^14 points
    (998244353, 18, 33, 17, 15000, 16200),  # 2^15
    (2013265921, 4, 33, 33, 35000, 5000),   # 2^16: column passes and blocks
    (469762049, 3, 33, 33, 60001, 7000),    # 2^17
    (998244353, 17, 32, 18, 24000, 3700),   # an operand below the line, the other over half the transform
    (998244353, 192, 4, 4, 8000, 8000),     # short strides: matfirst copied, matrowfirst operands not
    (268435399, 40, 36, 33, 4000, 4100),    # three FFT primes
])
def test_products(ctx, p, m, k, n, sa, sb):
    rng = np.random.default_rng(m * k * n + sa)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    ref = PolynomialMatrix(m, n, sa + sb - 1)
    say("in place, polfirst", p, m, k, n, sa, sb)
    PolynomialMatrixMulDomain(p, ctx).mul(ref, PolynomialMatrix.from_polfirst(a, m, k),
                                          PolynomialMatrix.from_polfirst(b, k, n))
    ref = ref.to_polfirst()
    assert check_by_evaluation(a, b, ref, p, m, k, n, sa, sb, sa + sb - 1, [int(rng.integers(1, p))])
    for method in METHODS:
        for la, lb, lc in BY_COEFFICIENT:
            C = PolynomialMatrix(m, n, sa + sb - 1, lc)
            say("in place", p, m, k, n, sa, sb, method, la, lb, lc)
            PolynomialMatrixMulDomain(p, ctx, method).mul(C, PolynomialMatrix.from_polfirst(a, m, k, la),
                                                          PolynomialMatrix.from_polfirst(b, k, n, lb))
            assert np.array_equal(C.to_polfirst(), ref)


@pytest.mark.parametrize("small_left", [True, False])
@pytest.mark.parametrize("p,m,k,n,hdeg", [
    (998244353, 64, 40, 36, 2000),   # 2^12 points: whole (plain) or split (INT8) transforms
    (998244353, 36, 33, 34, 8000),   # 2^14
    (2013265921, 8, 33, 33, 16400),  # 2^16: column passes and blocks
    (268435399, 64, 40, 36, 2000),   # three FFT primes
])
def test_middle_products(ctx, p, m, k, n, hdeg, small_left):
    rng = np.random.default_rng(m * k * n + hdeg)
    big = 2 * hdeg - 1
    sa, sb = (hdeg, big) if small_left else (big, hdeg)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    P = PolynomialMatrix(m, n, sa + sb - 1)
    say("in place, product of a middle product", p, m, k, n, sa, sb)
    PolynomialMatrixMulDomain(p, ctx).mul(P, PolynomialMatrix.from_polfirst(a, m, k),
                                          PolynomialMatrix.from_polfirst(b, k, n))
    ref = P.to_polfirst()[:, hdeg - 1:2 * hdeg - 1]
    for method in METHODS:
        for la, lb, lc in BY_COEFFICIENT:
            C = PolynomialMatrix(m, n, hdeg, lc)
            say("in place, middle product", p, m, k, n, sa, sb, method, la, lb, lc)
            PolynomialMatrixFFTMulDomain(p, ctx, method).midproduct(
                C, PolynomialMatrix.from_polfirst(a, m, k, la), PolynomialMatrix.from_polfirst(b, k, n, lb), small_left)
            assert np.array_equal(C.to_polfirst(), ref)
