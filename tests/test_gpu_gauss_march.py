"""Gaussian smearing of many (site, right-hand side) units marches along z;
few units take one thread per unit.  Both add the same products in the same
order, so a large batch equals its members smeared one by one, and a whole
large lattice equals its slices, bit for bit: right-hand-side counts that
divide neither a wavefront nor a plane, extents of 4 to 26, z segments of
unequal length, the first and the last slice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nrhs,t", [((10, 14, 6, 18), 9, -1), ((6, 4, 22, 28), 16, -1), ((16, 12, 10, 36), 2, -1),
                                      ((26, 22, 20, 4), 12, 3), ((24, 24, 18, 2), 13, 0)])
def test_march_equals_single_members(q, L, nrhs, t):
    print(f"march L={L} nrhs={nrhs} t={t}", flush=True)
    u = q.Gauge(L, boundaryT=-1, host=q.gen_gauge(L, 0.3, 5))
    x, y = q.Spinor(L, nrhs=nrhs), q.Spinor(L, nrhs=nrhs)
    x.gaussian(3)
    y.Gaussian_smearing(x, u, 3, 4.0, t=t)
    for r in (0, nrhs - 1):
        a, b = q.Spinor(L, host=x.download_rhs(r)), q.Spinor(L)
        b.Gaussian_smearing(a, u, 3, 4.0, t=t)
        assert np.array_equal(y.download_rhs(r), b.download()), r


def test_march_equals_slices(q):
    L = (16, 16, 16, 32)
    print(f"march L={L} against its slices", flush=True)
    u = q.Gauge(L, boundaryT=-1, host=q.gen_gauge(L, 0.3, 6))
    x, y, s = q.Spinor(L, host=q.gen_gaussian(L, 4)), q.Spinor(L), q.Spinor(L)
    y.Gaussian_smearing(x, u, 2, 4.0)
    got = y.download().reshape(L[3], -1)
    for t in (0, 13, 31):
        s.Gaussian_smearing(x, u, 2, 4.0, t=t)
        assert np.array_equal(got[t], s.download().reshape(L[3], -1)[t]), t
