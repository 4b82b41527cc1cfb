"""APE smearing on lattices that do not fill the last wavefront or workgroup
of its launch, against the oracle: rounding only (1e-12 after two steps, as
for the other short chains)."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 2), (6, 4, 6, 4), (6, 10, 6, 6), (12, 8, 10, 8)])
def test_ape_launch_shapes(q, L):
    print(f"APE L={L}", flush=True)
    U = q.gen_gauge(L, 0.25, 13)
    u, v = q.Gauge(L, boundaryT=-1, host=U), q.Gauge(L, boundaryT=-1)
    v.APE_smearing(u, 2, 0.5)
    assert np.max(np.abs(v.download() - orc.ape_smear(U, L, 2, 0.5))) <= 1e-12
