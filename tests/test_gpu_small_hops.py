"""FP64 hops of small lattices, whose directions run on eight wavefronts,
against the one-thread-per-site kernel, which a caller gets by asking for the
blocked walk or for a launch shape: every operator form, both bases and link
storages, on lattices whose parity does not fill its last 64 sites and on some
that take the XCD-remapped grid, with and without padding workgroups.  Both
kernels form and add the same FP64 products in the same order: the same bits,
and the bits of a batch's members."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (6, 4, 6, 4), (4, 6, 10, 6), (8, 8, 8, 16), (10, 8, 8, 14)])
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
        for name in ("split", "walk", "shape"):
            q.set_site_order(1 if name == "walk" else 2)
            q.set_tuning(block=128 if name == "shape" else 256)
            for op, run in ops.items():
                run()
                got[name, op] = (f if op == "normal_odd" else y).download()
    finally:
        q.set_site_order(2)
        q.set_tuning()
    for op in ops:
        assert np.array_equal(got["split", op], got["walk", op]) and np.array_equal(got["split", op], got["shape", op]), op
    b, c = q.Spinor(L, host=np.stack([psi, 2 * psi]), nrhs=2), q.Spinor(L, nrhs=2)
    c.tm(b, u, p)
    assert np.array_equal(c.download_rhs(0), got["split", "tm"])
