"""Batched hops on a lattice whose t slice exceeds an XCD's L2 walk the sites
in blocks by default: the same bits as in checkerboard order, for 8 (the
fewest) and 12 right-hand sides in every storage, with extents that 8 does not
divide."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,nrhs", [("HALF", 12), ("HALF", 8), ("BF16", 12), ("SINGLE", 8), ("SINGLE", 12),
                                       ("DOUBLE", 8)])
def test_batch_walk_identical(q, prec, nrhs):
    L = (20, 20, 22, 6)
    print(f"batch walk L={L} {prec} nrhs={nrhs}", flush=True)
    P = getattr(q, prec)
    u = q.Gauge(L, P, q.RECON_12, -1)
    u.convert_from(q.Gauge(L, boundaryT=-1, host=q.gen_gauge(L, 0.4, 2)))
    p = q.params(L, 0.156, 0.01, 1, -1)
    x, y = q.Spinor(L, P, q.EVEN, nrhs=nrhs), q.Spinor(L, P, q.EVEN, nrhs=nrhs)
    x.gaussian(7)
    got = {}
    try:
        q.set_autotune(0)
        for order in (0, 1, 2):
            q.set_site_order(order)
            y.tm_xxDagTm_xx(x, u, p, q.EE)
            got[order] = y.download()
    finally:
        q.set_site_order(2)
        q.set_autotune(1)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
