"""Learned preconditioner kernels at the edges of their launch shapes, against
the CPU oracle's layers: the even-odd network with per-thread links (up to 2
or 6 right-hand sides, by hidden channels) and links shared in LDS, workgroups
of 64, 128 and 256 threads, last workgroups partly empty and right-hand-side
counts that do not divide a wavefront; the gradient on lattices that do not fill
its last workgroup, on one that takes its 256-thread form and on one whose
workgroups go through more rounds of sites than their FP32 sums hold (9).

Tolerances: everything is FP32 arithmetic on FP32 data, so the network agrees
to a few roundings of its about 100-term sums (2e-6, as for the other FP32
operators) and the gradient, sums of up to 1e5 terms of either sign, to 1e-4."""
import numpy as np
import pytest

import oracle as orc
from refops import rel
from test_gpu_learned_solver import oracle_eo, rand_weights

pytestmark = pytest.mark.gpu


def _links(q, L, seed):
    U = q.gen_gauge(L, 0.4, seed)
    u32 = q.Gauge(L, q.SINGLE, q.RECON_18, -1)
    u32.convert_from(q.Gauge(L, boundaryT=-1, host=U))
    return u32, orc.apply_bc(U, L, -1)


@pytest.mark.parametrize("L,nrhs,ch", [((4, 6, 4, 6), 1, 4), ((4, 6, 4, 6), 2, 16), ((4, 6, 4, 6), 5, 4),
                                       ((6, 4, 6, 4), 7, 8), ((6, 4, 6, 4), 6, 4), ((6, 4, 6, 4), 7, 4),
                                       ((6, 4, 6, 4), 3, 8), ((6, 4, 6, 4), 16, 4), ((16, 12, 16, 16), 6, 4),
                                       ((20, 16, 20, 16), 3, 4), ((20, 16, 20, 16), 3, 8),
                                       ((24, 24, 24, 20), 1, 4)])
def test_net_eo_launch_shapes(q, L, nrhs, ch):
    print(f"N_e L={L} nrhs={nrhs} ch={ch}", flush=True)
    u32, Ub = _links(q, L, 17)
    W1, W2 = rand_weights(ch, 5)
    net = q.Net(ch, W1, W2)
    net.set_bf16(False)
    srcs = np.stack([q.gen_gaussian(L, 80 + r) for r in range(nrhs)])
    x = q.Spinor(L, q.SINGLE, q.EVEN, host=srcs, nrhs=nrhs)
    y = q.Spinor(L, q.SINGLE, q.EVEN, nrhs=nrhs)
    for adjoint in (False, True):
        net.apply_eo(y, x, u32, adjoint)
        got = y.download()
        got = got[None] if nrhs == 1 else got
        for r in {0, nrhs - 1}:
            assert rel(got[r], oracle_eo(srcs[r], Ub, L, W1, W2, adjoint)) <= 2e-6, (adjoint, r)


@pytest.mark.parametrize("L,ch", [((6, 4, 6, 6), 4), ((6, 4, 6, 6), 16), ((4, 4, 6, 10), 8), ((16, 12, 16, 16), 8),
                                  ((24, 22, 24, 18), 16)])
@pytest.mark.parametrize("prec", ["SINGLE", "DOUBLE"])
def test_net_gradient_launch_shapes(q, L, ch, prec):
    print(f"gradient L={L} ch={ch} {prec}", flush=True)
    u32, Ub = _links(q, L, 19)
    W1, W2 = rand_weights(ch, 6)
    net = q.Net(ch, W1, W2)
    net.set_bf16(False)
    P = getattr(q, prec)
    r, e = (q.gen_gaussian(L, s).astype(np.complex64).astype(np.complex128) for s in (1, 2))
    net.zero_grad()
    net.accumulate_grad(q.Spinor(L, P, host=r), q.Spinor(L, P, host=e), u32)
    G1, G2, loss = net.read_grad()
    ref, R1, R2 = orc.net_loss_grad(r, e, Ub, L, W1, W2)
    assert abs(loss - ref) <= 1e-5 * ref
    assert rel(G1, R1) <= 1e-4 and rel(G2, R2) <= 1e-4
