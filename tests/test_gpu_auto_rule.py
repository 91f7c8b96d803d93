"""AUTO on both sides of its lines below 2^12 points and above 2^15: the product is the
same as in either form by name, for one prime and for several (which share the line's
launches), checked by evaluation at a random point."""
import numpy as np
import pytest

import linbox_amd as lbx
from linbox_amd import PolynomialMatrix, PolynomialMatrixMulDomain
from polycheck import check_by_evaluation
from test_gpu_parity import ctx, rand, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,sa,sb", [
    (16, 16, 16, 1, 2), (16, 100, 17, 2, 1), (32, 512, 32, 1, 2), (33, 300, 30, 2, 3),   # 2 and 4 points
    (64, 64, 64, 16, 17), (40, 200, 33, 13, 20), (130, 140, 129, 16, 16),                # 32 points
    (16, 128, 16, 32, 33), (128, 512, 128, 64, 64),                                     # 64 and 128
    (96, 128, 96, 128, 128), (80, 100, 128, 127, 129), (64, 192, 64, 250, 260), (120, 64, 120, 256, 256),
    (112, 112, 112, 250, 263), (100, 64, 100, 512, 500), (128, 100, 128, 256, 257),
    (33, 17, 40, 33000, 9), (16, 16, 16, 32769, 20000),                                  # 2^16 points
])
@pytest.mark.parametrize("p", [998244353, 2013265921, 268435399])
def test_auto_agrees_with_both_forms(ctx, p, m, k, n, sa, sb):
    rng = np.random.default_rng(m * k * n + sa)
    a, b = rand(rng, p, m * k * sa).reshape(m * k, sa), rand(rng, p, k * n * sb).reshape(k * n, sb)
    a[:, 0], b[:, -1] = p - 1, p // 2
    got = []
    for method in (lbx.METHOD_AUTO, lbx.METHOD_PLAIN_U64, lbx.METHOD_INT8_MFMA):
        say("auto rule", p, m, k, n, sa, sb, method)
        C = PolynomialMatrix(m, n, sa + sb - 1)
        PolynomialMatrixMulDomain(p, ctx, method).mul(C, PolynomialMatrix.from_polfirst(a, m, k),
                                                      PolynomialMatrix.from_polfirst(b, k, n))
        got.append(C.to_polfirst())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    assert check_by_evaluation(a, b, got[0], p, m, k, n, sa, sb, sa + sb - 1, [int(rng.integers(1, p))])
