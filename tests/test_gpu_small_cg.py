"""The reference CG on small lattices -- the CG update fused into hops that run a
site's directions on eight wavefronts, partial sums of padding workgroups, and
the direction step of one thread per complex number up to 10,240 sites -- after
a fixed number of iterations against the oracle's, and against the kernels that
larger lattices take.

Twelve iterations apply the operator 24 times, 144-term FP64 sums each (about
1e-15), to directions whose coefficients carry the same errors; the recurrences
amplify them by less than the condition number, below 1e3 here: 1e-11."""
import numpy as np
import pytest

import oracle as orc
from refops import rel

pytestmark = pytest.mark.gpu
K, MU, ITERS = 0.156, 0.01, 12


@pytest.mark.parametrize("L", [(4, 4, 4, 2), (10, 8, 8, 14), (10, 8, 8, 16), (12, 10, 12, 10), (16, 8, 8, 16),
                               (12, 10, 14, 10)])
def test_fixed_iterations_match_oracle(q, L):
    print(f"CG L={L}", flush=True)
    U, b = q.gen_gauge(L, 0.4, 11), q.gen_gaussian(L, 12)
    u, bd = q.Gauge(L, boundaryT=-1, host=U), q.Spinor(L, host=b)
    p = q.params(L, K, MU, 1, -1, tol=1e-30, maxIter=ITERS)
    ref, k, _ = orc.cg(b, orc.apply_bc(U, L, -1), L, K, MU, 1, 1e-30, ITERS)
    assert k == ITERS
    x = {}
    try:
        for order in (2, 1):
            q.set_site_order(order)
            y = q.Spinor(L)
            st = q.CG(p, u)(y, bd)
            assert st.iterations == ITERS
            x[order] = y.download()
    finally:
        q.set_site_order(2)
    for order in (2, 1):
        assert rel(x[order], ref) <= 1e-11, order


def test_blocked_walk_reaches_small_lattices(q):
    """Asked for, the blocked walk is taken on small FP64 lattices too: it groups
    the partial sums differently, which shows in the last bits of an iterate (and
    no further: rounding amplified by the condition number over 60 iterations)."""
    L = (10, 8, 8, 14)
    u, b = q.Gauge(L, boundaryT=-1, host=q.gen_gauge(L, 0.4, 11)), q.Spinor(L, host=q.gen_gaussian(L, 12))
    x = {}
    try:
        for order in (2, 1):
            q.set_site_order(order)
            y = q.Spinor(L)
            q.CG(q.params(L, K, MU, 1, -1, tol=1e-30, maxIter=60), u)(y, b)
            x[order] = y.download()
    finally:
        q.set_site_order(2)
    assert not np.array_equal(x[1], x[2])
    assert rel(x[1], x[2]) <= 1e-9
