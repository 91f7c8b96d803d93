"""Plain products on transforms of several passes (2^16 points and more): the forward
transforms leave centred words and the pointwise stage takes its tiles, as it does for
whole transforms.  Every tile width and the split inner dimension at the edges of their
ranges, one prime and three, and a middle product; checked by evaluation at two points,
a middle product against the middle of the product."""
import numpy as np
import pytest

import linbox_amd as lbx
from linbox_amd import PolynomialMatrix, PolynomialMatrixFFTMulDomain, PolynomialMatrixMulDomain
from polycheck import check_by_evaluation
from test_gpu_parity import ctx, rand, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (3, 7, 4),     # 2x2 tiles
    (4, 9, 3), (2, 8, 4),     # 4x4 tiles, the inner dimension split
    (5, 3, 4), (8, 13, 7),    # 4x4 tiles
    (9, 5, 8), (17, 6, 10),   # 8x8 tiles with a remainder
])
@pytest.mark.parametrize("p,sa,sb", [(998244353, 32769, 32768), (2013265921, 60000, 5538), (998244353, 65537, 60000),
                                     (268435399, 33000, 32500)])
def test_long_plain_products(ctx, p, sa, sb, m, k, n):
    rng = np.random.default_rng(m * k * n + sa)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    a[:, 0], b[:, 0], a[0], b[-1] = p // 2, p // 2 + 1, p // 2, p - 1
    C = PolynomialMatrix(m, n, sa + sb - 1)
    say("long plain product", p, m, k, n, sa, sb)
    PolynomialMatrixMulDomain(p, ctx, lbx.METHOD_PLAIN_U64).mul(C, PolynomialMatrix.from_polfirst(a, m, k),
                                                               PolynomialMatrix.from_polfirst(b, k, n))
    xs = [int(x) for x in rng.integers(0, p, 2)]
    assert check_by_evaluation(a, b, C.to_polfirst(), p, m, k, n, sa, sb, sa + sb - 1, xs)


@pytest.mark.parametrize("small_left", [True, False])
@pytest.mark.parametrize("p", [998244353, 268435399])
def test_long_plain_middle_product(ctx, p, small_left):
    m, k, n, hdeg = 9, 9, 5, 33000
    sa, sb = (hdeg, 2 * hdeg - 1) if small_left else (2 * hdeg - 1, hdeg)
    rng = np.random.default_rng(hdeg)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    A, B = PolynomialMatrix.from_polfirst(a, m, k), PolynomialMatrix.from_polfirst(b, k, n)
    P, C = PolynomialMatrix(m, n, sa + sb - 1), PolynomialMatrix(m, n, hdeg)
    say("long plain middle product", p, small_left)
    PolynomialMatrixMulDomain(p, ctx, lbx.METHOD_PLAIN_U64).mul(P, A, B)
    PolynomialMatrixFFTMulDomain(p, ctx, lbx.METHOD_PLAIN_U64).midproduct(C, A, B, small_left)
    assert np.array_equal(C.to_polfirst(), P.to_polfirst()[:, hdeg - 1:2 * hdeg - 1])


@pytest.mark.parametrize("m,k,n", [(1, 64, 64), (2, 30, 60), (60, 5, 2), (35, 7, 4), (4, 9, 70), (5, 3, 40), (60, 2, 3)])
@pytest.mark.parametrize("p,sa,sb", [(998244353, 8193, 8000), (2013265921, 16384, 16385), (268435399, 4000, 4097)])
def test_narrow_plain_products(ctx, p, sa, sb, m, k, n):
    """Products of few rows or columns on transforms that fill the chip: tiles no wider
    than the narrow side needs, whole transforms and those of several passes."""
    rng = np.random.default_rng(m * k * n + sa)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    a[0], b[-1] = p // 2, p - 1
    C = PolynomialMatrix(m, n, sa + sb - 1)
    say("narrow plain product", p, m, k, n, sa, sb)
    PolynomialMatrixMulDomain(p, ctx, lbx.METHOD_PLAIN_U64).mul(C, PolynomialMatrix.from_polfirst(a, m, k),
                                                               PolynomialMatrix.from_polfirst(b, k, n))
    assert check_by_evaluation(a, b, C.to_polfirst(), p, m, k, n, sa, sb, sa + sb - 1, [int(rng.integers(1, p))])
