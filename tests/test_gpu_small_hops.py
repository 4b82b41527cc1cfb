"""FP64 hops of small lattices, whose directions run on eight wavefronts,
against the one-thread-per-site kernel (which the autotuner, asked to tune
every launch, selects): every operator form, both bases and link storages, on
lattices whose parity does not fill its last 64 sites and on one that takes
the XCD-remapped grid.  Both kernels form and add the same FP64 products in
the same order; the compiler may contract one product and sum differently, so
the results may differ in the last bits of a hop's 144-term sums (1e-15)."""
import numpy as np
import pytest

from refops import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (6, 4, 6, 4), (4, 6, 10, 6), (8, 8, 8, 16)])
@pytest.mark.parametrize("recon", ["RECON_18", "RECON_12"])
def test_split_hop_matches_one_thread_per_site(q, L, recon):
    print(f"split hops L={L} {recon}", flush=True)
    U = q.gen_gauge(L, 0.4, 3)
    u = q.Gauge(L, q.DOUBLE, getattr(q, recon), -1, host=U)
    p = q.params(L, 0.156, 0.02, 1, -1)
    psi = q.gen_gaussian(L, 4)
    x, y = q.Spinor(L, host=psi), q.Spinor(L)
    e, f = q.Spinor(L, q.DOUBLE, q.ODD, host=psi), q.Spinor(L, q.DOUBLE, q.ODD)
    ops = {
        "hop": lambda: y.applyDslash(x, u), "hop_dag": lambda: y.applyDslashDag(x, u),
        "hop_chiral": lambda: y.applyDslash(x, u, q.CHIRAL), "tm": lambda: y.tm(x, u, p),
        "tm_chiral": lambda: y.tm(x, u, p, q.CHIRAL), "tmDag": lambda: y.tmDag(x, u, p),
        "Wilson": lambda: y.Wilson(x, u, p), "tm_xx": lambda: y.tm_xx(x, u, p, q.EE),
        "tm_xx_chiral": lambda: y.tm_xx(x, u, p, q.OO, q.CHIRAL),
        "normal_odd": lambda: f.tm_xxDagTm_xx(e, u, p, q.OO),
    }
    got = {}
    try:
        for mode in (2, 0):
            q.set_autotune(mode)
            for name, run in ops.items():
                run()
                got[name, mode] = (f if name == "normal_odd" else y).download()
    finally:
        q.set_autotune(1)
    for name in ops:
        assert rel(got[name, 0], got[name, 2]) <= 1e-15, name
