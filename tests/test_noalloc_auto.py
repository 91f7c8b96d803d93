"""AUTO through lbx_polymat_mul_u32_noalloc where its faster form needs more than the
64 MiB of the fixed workspace and the other one fits: the product is formed in that
one, and equals the allocating entry point's."""
import numpy as np
import pytest

import linbox_amd as lbx
from test_zz_no_alloc import ctx, run_both, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,m,k,n,sa,sb", [
    (998244353, 90, 128, 90, 256, 257),   # 61 MiB plain, 86 INT8
    (2013265921, 64, 192, 64, 200, 250),  # 56, 80
    (998244353, 120, 64, 120, 250, 263),  # 58, 88
])
def test_auto_fits_where_plain_does(ctx, p, m, k, n, sa, sb):
    say("noalloc auto", p, m, k, n, sa, sb)
    plain = run_both(ctx, p, m, k, n, sa, sb, lbx.METHOD_PLAIN_U64, seed=m)
    want, got = run_both(ctx, p, m, k, n, sa, sb, lbx.METHOD_AUTO, seed=m)
    assert np.array_equal(got, want) and np.array_equal(got, plain[1])
