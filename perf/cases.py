"""Performance cases: the work a user of qkxtm_mpi_amd has it do.

Each case is one call, or one short chain of calls, of the package's public
interface on fields that stay on the GPU, as in the examples and the studies
of bench.py:

  operator   Dirac operator: the full twisted-mass operator (tm), or the normal
             even-odd operator (tm_xxDagTm_xx) that every solver iterates, on
             one right-hand side or a batch, in each storage precision
  cg         reference conjugate gradient, FP64
  solve      even-odd mixed-precision solve of one source
  propagator lockstep solve of a batch of spin-colour point sources
  ape        APE smearing of the links
  gauss      Gaussian smearing of a batch of sources (one time slice) or of
             sinks (whole lattice)
  net        learned preconditioner, forward and adjoint, inside a solve
  train      gradient of the learned preconditioner over a few random pairs

Outputs are read in place: a field's device memory is viewed as a torch
tensor, component-major over parity-blocked sites (the layout stated at the
top of qkx_internal.h), so a pass copies nothing to the host that the call
itself does not.

`exact` restates each path in 64-bit torch on the whole lattice, from the
definitions of the operators.
"""
import ctypes
import math

import numpy as np
import torch

import qkxtm_mpi_amd as q

PREC = {"double": q.DOUBLE, "single": q.SINGLE, "half": q.HALF, "bf16": q.BF16}
DELTA = {"single": 0.003, "half": 0.003, "bf16": 0.03}   # bench.py's reliable-update triggers
TOL = 1e-10
ALPHA_APE, ALPHA_GAUSS = 0.5, 4.0                        # bin/test_gauss_smearing.cpp:31-34
CAP = {"operator": 2 << 20, "cg": 40000, "solve": 680000, "propagator": 140000, "ape": 1 << 20, "gauss": 680000,
       "net": 680000, "train": 140000}                   # most sites of a drawn case
LEAST = {"operator": 512, "cg": 512, "solve": 8192, "propagator": 8192, "ape": 2048, "gauss": 2048, "net": 2048,
         "train": 2048}


def listed():
    return [
        # one application of the drop-in operator on the smallest lattice of
        # the examples: launch latency
        dict(name="tm_small", kind="operator", form="tm", prec="double", nrhs=1, x=8, y=8, z=8, t=16),
        # the headline lattice's operator, device resident, FP64
        dict(name="tm_headline", kind="operator", form="tm", prec="double", nrhs=1, x=24, y=24, z=24, t=48),
        # what the FP16 solver of the headline lattice iterates
        dict(name="normal_half", kind="operator", form="normal", prec="half", nrhs=1, x=24, y=24, z=24, t=48),
        # what a 12-source propagator solve iterates, at the batched study's volume
        dict(name="normal_half_batch", kind="operator", form="normal", prec="half", nrhs=12, x=32, y=32, z=32, t=64),
        # three twisted masses at once, FP32 inner, on a lattice of unequal sides
        dict(name="normal_single_ragged", kind="operator", form="normal", prec="single", nrhs=3, x=20, y=12, z=28,
             t=36),
        # the reference algorithm on the plain-method example: FP64 CG at 8^3x16
        dict(name="cg_reference", kind="cg", x=8, y=8, z=8, t=16, kappa=0.156, mu=0.01, eps=0.4),
        # the headline: one source to a true residual of 1e-10, FP16 inner
        dict(name="solve_headline", kind="solve", prec="half", x=24, y=24, z=24, t=48, kappa=0.1632, mu=0.004,
             eps=0.3),
        # a propagator: its 12 point sources in one batch
        dict(name="propagator", kind="propagator", prec="half", nrhs=12, x=16, y=16, z=16, t=32, kappa=0.1625,
             mu=0.004, eps=0.3),
        # smearing of a configuration before the solves
        dict(name="ape", kind="ape", steps=4, x=24, y=24, z=24, t=48),
        # smearing of the 12 solutions at the sink
        dict(name="gauss_sink", kind="gauss", steps=5, nrhs=12, slice=False, x=24, y=24, z=24, t=48),
        # the learned preconditioner of a 12-source batch: forward and adjoint
        dict(name="net_batch", kind="net", prec="half", ch=4, nrhs=12, x=24, y=24, z=24, t=48),
        # training of the 4 -> 16 -> 4 network on its lattice: four pairs
        dict(name="train", kind="train", ch=16, pairs=4, x=16, y=16, z=16, t=32),
    ]


def draw(rng):
    kind = rng.choice(["operator"] * 4 + ["cg", "solve", "propagator", "ape", "gauss", "gauss", "net", "train"])
    c = dict(kind=kind)
    cap = CAP[kind]
    if kind == "operator":
        c["form"] = rng.choice(["tm", "normal"])
        c["prec"] = rng.choice(["double", "single", "half", "half", "bf16"])
        c["nrhs"] = rng.choice([1, 1, 3, 12, rng.randint(2, 16)])
        cap = min(cap, (4 << 20) // c["nrhs"] if c["prec"] == "double" else (12 << 20) // c["nrhs"])
    elif kind == "cg":
        c.update(kappa=0.156, mu=0.01, eps=0.4)
    elif kind == "solve":
        c.update(prec=rng.choice(["half", "half", "single", "bf16"]), kappa=0.16, mu=rng.choice([0.004, 0.01, 0.02]),
                 eps=0.3)
    elif kind == "propagator":
        c.update(prec=rng.choice(["half", "half", "single"]), nrhs=rng.choice([3, 12, 12, rng.randint(2, 16)]),
                 kappa=0.16, mu=0.004, eps=0.3)
    elif kind == "ape":
        c["steps"] = rng.randint(1, 6)
    elif kind == "gauss":
        c["slice"] = rng.random() < 0.5
        c["nrhs"] = rng.choice([1, 3, 4, 12, 12])
        c["steps"] = rng.randint(10, 50) if c["slice"] else rng.randint(2, 5)
    elif kind == "net":
        c.update(prec=rng.choice(["half", "single", "bf16"]), ch=rng.choice([4, 4, 8, 16]),
                 nrhs=rng.choice([1, 4, 12, rng.randint(2, 16)]))
        cap = min(cap, 8 * 680000 // (c["nrhs"] * c["ch"] // 4) // 2)
    else:
        c.update(ch=rng.choice([4, 8, 16]), pairs=rng.randint(1, 4))
    # an even extent in each direction, spatial sides near each other, t longer
    while True:
        v = math.exp(rng.uniform(math.log(LEAST[kind]), math.log(cap)))
        s = (v / 2) ** 0.25
        side = [max(4, 2 * round(s * rng.uniform(0.75, 1.3) / 2)) for _ in range(3)]
        t = max(4, 2 * round(v / (side[0] * side[1] * side[2]) / 2))
        if LEAST[kind] <= side[0] * side[1] * side[2] * t <= cap and t <= 96:
            break
    c.update(x=side[0], y=side[1], z=side[2], t=t)
    return c


# ---- fields ---------------------------------------------------------------------------
class _Field(ctypes.Structure):
    """The head of a spinor field's handle."""
    _fields_ = [("L", ctypes.c_int * 4), ("V", ctypes.c_int), ("Vh", ctypes.c_int), ("prec", ctypes.c_int),
                ("subset", ctypes.c_int), ("nsites", ctypes.c_int), ("nrhs", ctypes.c_int), ("data", ctypes.c_void_p),
                ("nrm", ctypes.c_void_p)]


class _Links(ctypes.Structure):
    """The head of a gauge field's handle."""
    _fields_ = [("L", ctypes.c_int * 4), ("V", ctypes.c_int), ("Vh", ctypes.c_int), ("prec", ctypes.c_int),
                ("recon", ctypes.c_int), ("bc", ctypes.c_int), ("data", ctypes.c_void_p)]


class _Memory:
    """Device memory of a field, for torch; keeps the field alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, ptr, shape, typestr):
    return torch.as_tensor(_Memory(owner, ptr, shape, typestr), device="cuda")


def spinor_view(f):
    """The stored arrays of a spinor field: [values], or [values, scales] in half precision."""
    h = ctypes.cast(f.h, ctypes.POINTER(_Field)).contents
    n = h.nsites * h.nrhs
    if h.prec == q.DOUBLE:
        return [_tensor(f, h.data, (12, n, 2), "<f8")]
    if h.prec == q.SINGLE:
        return [_tensor(f, h.data, (6, n, 4), "<f4")]
    if h.prec == q.HALF:
        return [_tensor(f, h.data, (3, n, 8), "<f2"), _tensor(f, h.nrm, (n,), "<f4")]
    return [_tensor(f, h.data, (3, n, 8), "<i2").view(torch.bfloat16)]


def gauge_view(u):
    h = ctypes.cast(u.h, ctypes.POINTER(_Links)).contents
    return _tensor(u, h.data, (36, h.V, 2), "<f8")


def shape_of(case):
    return (case["x"], case["y"], case["z"], case["t"])


def site_order(L):
    """Lexicographic site index (x fastest) of each parity-blocked site."""
    x, y, z, t = (torch.arange(n, device="cuda") for n in L)
    par = (t[:, None, None, None] + z[None, :, None, None] + y[None, None, :, None] + x[None, None, None, :]) & 1
    par = par.reshape(-1)
    lex = torch.arange(par.numel(), device="cuda")
    return torch.cat([lex[par == 0], lex[par == 1]])


def stored(psi, L, prec, subset=q.FULL):
    """The arrays that hold `psi` [V, nrhs, 4, 3] (lexicographic, complex128), as spinor_view lays them out, in 64 bits."""
    order = site_order(L)
    if subset == q.EVEN:
        order = order[: order.numel() // 2]
    v = torch.view_as_real(psi[order].reshape(-1, 12))           # [entries, 12, 2]
    if prec == "double":
        return [v.permute(1, 0, 2)]
    if prec == "single":
        return [v.reshape(-1, 6, 4).permute(1, 0, 2)]
    v = v.reshape(-1, 3, 8)
    if prec == "bf16":
        return [v.permute(1, 0, 2)]
    m = v.abs().amax((1, 2))
    return [(v / m.clamp_min(1e-300)[:, None, None]).permute(1, 0, 2), m]


def new_spinor(L, prec="double", subset=q.FULL, nrhs=1, psi=None):
    f = q.Spinor(L, PREC[prec], subset, nrhs=nrhs)
    if psi is None:
        f.zero()
    else:
        for a, b in zip(spinor_view(f), stored(psi, L, prec, subset)):
            a.copy_(b)
    return f


# ---- inputs, from the seed alone --------------------------------------------------------
def _normal(gen, *shape):
    return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, device="cuda", dtype=torch.float64))


def generator(seed, what):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + what)


def mm(a, b):
    """a b of small matrices stored in the last two dimensions."""
    return sum(a[..., :, k, None] * b[..., k, None, :] for k in range(a.shape[-1]))


def dag(a):
    return a.conj().transpose(-1, -2)


def conj_cross(a, b):
    return torch.stack([(a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1]).conj(),
                        (a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2]).conj(),
                        (a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]).conj()], -1)


def links(L, eps, seed):
    """U = exp(i eps H) reunitarised to SU(3), H Hermitian and traceless with Gaussian entries: [T, Z, Y, X, 4, 3, 3]."""
    a = _normal(generator(seed, 1), L[3], L[2], L[1], L[0], 4, 3, 3)
    h = 0.5 * (a + dag(a))
    eye = torch.eye(3, dtype=h.dtype, device=h.device)
    h = h - (h.diagonal(dim1=-2, dim2=-1).sum(-1) / 3)[..., None, None] * eye
    x, e = 1j * eps * h, 0
    for n in range(8, 0, -1):
        e = mm(x, eye + e) / n
    e = eye + e
    r0 = e[..., 0, :] / e[..., 0, :].abs().square().sum(-1, keepdim=True).sqrt()
    r1 = e[..., 1, :]
    for _ in range(2):
        r1 = r1 - (r0.conj() * r1).sum(-1, keepdim=True) * r0
        r1 = r1 / r1.abs().square().sum(-1, keepdim=True).sqrt()
    return torch.stack([r0, r1, conj_cross(r0, r1)], -2)


def upload_links(L, U, prec=None):
    """FP64 links with an antiperiodic time boundary, and their copy for fields of `prec`."""
    u = q.Gauge(L, q.DOUBLE, q.RECON_18, -1, host=U.reshape(-1, 4, 3, 3).cpu().numpy())
    if prec is None or prec == "double":
        return u, u
    v = q.Gauge(L, PREC[prec], q.RECON_12, -1)
    v.convert_from(u)
    return u, v


def gaussian(L, nrhs, seed):
    return _normal(generator(seed, 2), L[0] * L[1] * L[2] * L[3], nrhs, 4, 3)


def z2(L, nrhs, seed):
    b = torch.randint(0, 2, (L[0] * L[1] * L[2] * L[3], nrhs, 4, 3, 2), generator=generator(seed, 3), device="cuda")
    return torch.view_as_complex((2.0 * b.to(torch.float64) - 1.0) / math.sqrt(2.0))


def point_site(L, seed):
    g = torch.Generator().manual_seed(int(seed) + 4)
    return [int(torch.randint(0, n, (1,), generator=g)) for n in L]


def points(L, nrhs, seed):
    """Spin-colour point sources at one site; past the twelfth, at the next sites."""
    x0 = point_site(L, seed)
    V = L[0] * L[1] * L[2] * L[3]
    iv = ((x0[3] * L[2] + x0[2]) * L[1] + x0[1]) * L[0] + x0[0]
    psi = torch.zeros(V, nrhs, 4, 3, dtype=torch.complex128, device="cuda")
    for r in range(nrhs):
        psi[(iv + r // 12) % V, r, (r % 12) // 3, r % 3] = 1.0
    return psi


def weights(ch, seed):
    """A network near the identity, as training starts and leaves it: W1 [9, ch, 4], W2 [9, 4, ch]."""
    g = torch.Generator().manual_seed(int(seed) + 5)
    w = 0.05 * torch.randn(2, 9, ch, 4, 2, generator=g, dtype=torch.float64)
    W1 = torch.view_as_complex(w[0].contiguous())
    W2 = torch.view_as_complex(w[1].contiguous()).transpose(1, 2).contiguous()
    W1[0, :4, :4] += torch.eye(4)
    W2[0, :4, :4] += torch.eye(4)
    return W1.numpy(), W2.numpy()


# ---- prepare and run --------------------------------------------------------------------
KAPPA, MU, EPS = 0.1632, 0.004, 0.3


def prepare(case, seed):
    L, kind = shape_of(case), case["kind"]
    s = {"case": case}
    U = links(L, case.get("eps", EPS), seed)
    p = q.params(L, case.get("kappa", KAPPA), case.get("mu", MU), 1, -1, tol=TOL, maxIter=20000)
    s["p"] = p
    if kind == "operator":
        s["u64"], s["u"] = upload_links(L, U, case["prec"])
        sub = q.EVEN if case["form"] == "normal" else q.FULL
        s["in"] = new_spinor(L, case["prec"], sub, case["nrhs"], gaussian(L, case["nrhs"], seed))
        s["out"] = new_spinor(L, case["prec"], sub, case["nrhs"])
    elif kind in ("cg", "solve"):
        s["u"], _ = upload_links(L, U)
        s["in"] = new_spinor(L, psi=z2(L, 1, seed))
        s["out"] = new_spinor(L)
    elif kind == "propagator":
        s["u"], _ = upload_links(L, U)
        s["in"] = new_spinor(L, nrhs=case["nrhs"], psi=points(L, case["nrhs"], seed))
        s["out"] = new_spinor(L, nrhs=case["nrhs"])
    elif kind == "ape":
        s["u"], _ = upload_links(L, U)
        s["out"] = q.Gauge(L, q.DOUBLE, q.RECON_18, -1)
    elif kind == "gauss":
        s["u"], _ = upload_links(L, U)
        src = points(L, case["nrhs"], seed) if case["slice"] else gaussian(L, case["nrhs"], seed)
        s["in"] = new_spinor(L, nrhs=case["nrhs"], psi=src)
        s["out"] = new_spinor(L, nrhs=case["nrhs"])
        s["t"] = point_site(L, seed)[3] if case["slice"] else -1
    else:
        u, _ = upload_links(L, U)
        s["u"] = q.Gauge(L, q.SINGLE, q.RECON_18, -1)
        s["u"].convert_from(u)
        s["net"] = q.Net(case["ch"], *weights(case["ch"], seed))
        if kind == "net":
            s["in"] = new_spinor(L, case["prec"], q.EVEN, case["nrhs"], gaussian(L, case["nrhs"], seed))
            s["mid"] = new_spinor(L, case["prec"], q.EVEN, case["nrhs"])
            s["out"] = new_spinor(L, case["prec"], q.EVEN, case["nrhs"])
        else:
            s["e"] = [new_spinor(L, "single", psi=e) for e in pairs_of(case, seed)]
            s["r"] = new_spinor(L, "single")
    # the views of what run() returns; the fields are made once, as in a program's loop
    if kind == "ape":
        s["view"] = gauge_view(s["out"])
    elif kind != "train":
        s["view"] = [spinor_view(s[k]) for k in (("mid", "out") if kind == "net" else ("out",))]
    torch.cuda.synchronize()   # the library runs on a stream of its own
    return s


def pairs_of(case, seed):
    """Unit-norm random error fields, rounded to FP32 as the network trains on them."""
    L = shape_of(case)
    out = []
    for k in range(case["pairs"]):
        e = gaussian(L, 1, 101 * int(seed) + k)
        e = e / e.abs().square().sum().sqrt()
        out.append(e.to(torch.complex64).to(torch.complex128))
    return out


def run(s):
    case, p = s["case"], s["p"]
    kind = case["kind"]
    if kind == "operator":
        if case["form"] == "tm":
            s["out"].tm(s["in"], s["u"], p)
        else:
            s["out"].tm_xxDagTm_xx(s["in"], s["u"], p, q.EE)
    elif kind == "cg":
        s["out"].zero()                       # the reference CG adds to its solution field
        q.CG(p, s["u"])(s["out"], s["in"])
    elif kind == "solve":
        q.solve(s["out"], s["in"], s["u"], p, eo=True, inner_prec=PREC[case["prec"]], delta=DELTA[case["prec"]],
                tol=TOL)
    elif kind == "propagator":
        q.solve_batch(s["out"], s["in"], s["u"], p, eo=True, inner_prec=PREC[case["prec"]],
                      delta=DELTA[case["prec"]], tol=TOL)
    elif kind == "ape":
        s["out"].APE_smearing(s["u"], case["steps"], ALPHA_APE)
    elif kind == "gauss":
        s["out"].Gaussian_smearing(s["in"], s["u"], case["steps"], ALPHA_GAUSS, t=s["t"])
    elif kind == "net":
        s["net"].apply_eo(s["mid"], s["in"], s["u"])
        s["net"].apply_eo(s["out"], s["mid"], s["u"], adjoint=True)
    else:
        net = s["net"]
        net.zero_grad()
        for e in s["e"]:
            s["r"].tm(e, s["u"], p)           # the pair (D e, e)
            net.accumulate_grad(s["r"], e, s["u"])
        g1, g2, loss = net.read_grad()
        return {"grad1": g1.astype(np.complex64), "grad2": g2.astype(np.complex64), "loss": np.float32(loss)}
    return s["view"]


# ---- what a pass cannot do without --------------------------------------------------------
SPINOR = {"double": 192, "single": 96, "half": 52, "bf16": 48}     # bytes of one site
LINK = {"double": 96, "single": 48, "half": 24, "bf16": 24}        # bytes of one link: two rows
HOP_FLOPS = 1320                                                   # of one site's eight-direction stencil


def work(case):
    """Inputs read once, outputs written once; the arithmetic of the definitions.  A solve counts the iterations that
    conjugate gradient takes on these systems (about 55 on the even-odd ones, 160 for the reference's), each of which has
    to pass over the links and over its vectors in the inner precision."""
    x, y, z, t = shape_of(case)
    V, kind = x * y * z * t, case["kind"]
    n = case.get("nrhs", 1)
    if kind == "operator":
        sites = V if case["form"] == "tm" else V // 2
        hops = 1 if case["form"] == "tm" else 4
        return {"bytes": 4.0 * V * LINK[case["prec"]] + 2.0 * sites * n * SPINOR[case["prec"]],
                "flops": (HOP_FLOPS + 96.0) * sites * n * hops}
    if kind == "cg":
        its, w = 160, 192.0
        return {"bytes": its * V * (4.0 * 96 + 6 * w), "flops": its * V * (2 * (HOP_FLOPS + 96.0) + 144)}
    if kind in ("solve", "propagator"):
        its, w = 55, float(SPINOR[case["prec"]])
        return {"bytes": its * V * (4.0 * LINK[case["prec"]] + 3 * n * w) + 2.0 * V * n * 192 + 4 * 96.0 * V,
                "flops": its * V / 2 * n * (4 * (HOP_FLOPS + 96.0) + 144)}
    if kind == "ape":
        return {"bytes": 2.0 * V * 4 * 144, "flops": case["steps"] * 3.0 * V * (8 * 198 + 1000)}
    if kind == "gauss":
        sites = V // t if case["slice"] else V
        return {"bytes": 3.0 * sites * 144 + 2.0 * sites * n * 192,
                "flops": case["steps"] * sites * n * (6.0 * 4 * 66 + 14 * 12)}
    ch = case["ch"]
    mix, hop = 8.0 * 4 * ch * 3, 8.0 * 4 * 66              # of one site: mixing by one path, transports by eight
    if kind == "net":
        return {"bytes": 2 * (4.0 * V * 72 + V * n * SPINOR[case["prec"]]),
                "flops": 2.0 * V / 2 * n * (2 * (8 * mix + hop) + 8 * 48)}
    return {"bytes": case["pairs"] * V * (4.0 * 72 + 96), "flops": case["pairs"] * V * (HOP_FLOPS + 5.0 * (9 * mix + hop))}


# ---- the definitions in 64 bits ------------------------------------------------------------
def _gammas():
    g = torch.zeros(5, 4, 4, dtype=torch.complex128, device="cuda")
    for mu, row in enumerate([[(0, 3, 1j), (1, 2, 1j), (2, 1, -1j), (3, 0, -1j)],
                              [(0, 3, 1), (1, 2, -1), (2, 1, -1), (3, 0, 1)],
                              [(0, 2, 1j), (1, 3, -1j), (2, 0, -1j), (3, 1, 1j)],
                              [(0, 0, 1), (1, 1, 1), (2, 2, -1), (3, 3, -1)],
                              [(0, 2, 1), (1, 3, 1), (2, 0, 1), (3, 1, 1)]]):
        for a, b, v in row:
            g[mu, a, b] = v
    return g


class Exact:
    """Fields [T, Z, Y, X, channels, 3] with links [T, Z, Y, X, 4, 3, 3]; antiperiodic in t."""

    def __init__(self, L, U):
        self.L, self.g = L, _gammas()
        self.U = U.clone()
        self.U[-1, ..., 3, :, :] *= -1
        self.Ub = torch.stack([dag(torch.roll(self.U[..., m, :, :], 1, 3 - m)) for m in range(4)], -3)

    def field(self, psi):
        x, y, z, t = self.L
        return psi.reshape(t, z, y, x, 4, 3)

    def transport(self, psi, path):
        """path 0: psi; 1 + 2 mu: U_mu(x) psi(x + mu); 2 + 2 mu: U_mu(x - mu)^dag psi(x - mu)."""
        if path == 0:
            return psi
        mu, back = (path - 1) // 2, (path - 1) % 2
        v = torch.roll(psi, 1 if back else -1, 3 - mu)
        W = (self.Ub if back else self.U)[..., mu, :, :]
        return sum(W[..., None, :, b] * v[..., :, b, None] for b in range(3))

    def spin(self, G, psi):
        out = torch.zeros_like(psi)
        for a in range(4):
            for b in range(4):
                if G[a, b] != 0:
                    out[..., a, :] += G[a, b] * psi[..., b, :]
        return out

    def hop(self, psi, dagger=False):
        one, out = torch.eye(4, dtype=psi.dtype, device=psi.device), 0
        for mu in range(4):
            for back in (0, 1):
                sign = -1 if back == (1 if dagger else 0) else 1
                # the spin matrix before the transport: it acts on another index
                out = out + self.transport(self.spin(one + sign * self.g[mu], psi), 1 + 2 * mu + back)
        return out

    def g5(self, psi):
        return psi[..., [2, 3, 0, 1], :]

    def tm(self, psi, kappa, mu, dagger=False):
        a = (-1 if dagger else 1) * 2 * kappa * mu
        return psi + 1j * a * self.g5(psi) - kappa * self.hop(psi, dagger)

    def even(self, psi):
        x, y, z, t = (torch.arange(n, device="cuda") for n in self.L)
        par = (t[:, None, None, None] + z[None, :, None, None] + y[None, None, :, None] + x[None, None, None, :]) & 1
        return psi * (par == 0)[..., None, None]

    def schur(self, psi, kappa, a):
        """On a field that is zero on the odd sites."""
        h = self.hop(psi)
        h = (h - 1j * a * self.g5(h)) / (1 + a * a)
        return self.even(psi + 1j * a * self.g5(psi) - kappa * kappa * self.hop(h))

    def normal(self, psi, kappa, mu):
        a = 2 * kappa * mu
        return self.g5(self.schur(self.g5(self.schur(psi, kappa, a)), kappa, -a))

    def solve(self, b, kappa, mu, normal):
        """D x = b, or D^dag D x = b (normal), to a residual near rounding."""
        rhs = b if normal else self.tm(b, kappa, mu, True)
        x, r = torch.zeros_like(b), rhs.clone()
        p, r2 = r.clone(), float(r.abs().square().sum())
        stop = 1e-28 * r2
        for _ in range(2000):
            dp = self.tm(p, kappa, mu)
            ap = self.tm(dp, kappa, mu, True)
            alpha = r2 / float(dp.abs().square().sum())
            x += alpha * p
            r -= alpha * ap
            new = float(r.abs().square().sum())
            if new <= stop:
                break
            p = r + (new / r2) * p
            r2 = new
        return x

    def layer(self, W, f):
        out = 0
        for path in range(9):
            v = self.transport(f, path)
            out = out + sum(W[path][:, b, None] * v[..., b, None, :] for b in range(v.shape[-2]))
        return out

    def layer_dag(self, W, f):
        rev = [0] + [p + 1 if p % 2 else p - 1 for p in range(1, 9)]
        return self.layer([dag(W[rev[p]]) for p in range(9)], f)


def _project(M):
    """SU(3) part of M: its polar factor without the phase of its determinant."""
    X = M
    for _ in range(12):
        cof = torch.stack([conj_cross(X[..., 1, :], X[..., 2, :]), conj_cross(X[..., 2, :], X[..., 0, :]),
                           conj_cross(X[..., 0, :], X[..., 1, :])], -2)       # conjugated cofactors
        det = (X[..., 0, :] * cof[..., 0, :].conj()).sum(-1)
        X = 0.5 * (X + cof / det.conj()[..., None, None])
    cof = conj_cross(X[..., 1, :], X[..., 2, :])
    det = (X[..., 0, :] * cof.conj()).sum(-1)
    return X * torch.polar(torch.ones_like(det.real), -det.angle() / 3)[..., None, None]


def _ape(U, steps):
    for _ in range(steps):
        new = U.clone()
        for mu in range(3):
            S = 0
            for nu in range(3):
                if nu == mu:
                    continue
                m, n = U[..., mu, :, :], U[..., nu, :, :]
                S = S + mm(mm(n, torch.roll(m, -1, 3 - nu)), dag(torch.roll(n, -1, 3 - mu)))
                down = mm(mm(dag(n), m), torch.roll(n, -1, 3 - mu))
                S = S + torch.roll(down, 1, 3 - nu)
            new[..., mu, :, :] = _project(U[..., mu, :, :] + ALPHA_APE * S)
        U = new
    return U


def _bf16(w):
    t = torch.from_numpy(np.ascontiguousarray(w.astype(np.complex64)).view(np.float32)).to(torch.bfloat16)
    return torch.view_as_complex(t.to(torch.float64).reshape(*w.shape, 2)).cuda()


def exact(case, seed):
    L, kind = shape_of(case), case["kind"]
    U = links(L, case.get("eps", EPS), seed)
    V, n = L[0] * L[1] * L[2] * L[3], case.get("nrhs", 1)
    kappa, mu = case.get("kappa", KAPPA), case.get("mu", MU)
    if kind == "ape":
        S = _ape(U, case["steps"])
        return torch.view_as_real(S.reshape(V, 36)[site_order(L)]).permute(1, 0, 2)
    E = Exact(L, U)
    if kind == "train":
        W1, W2 = (_bf16(w) for w in weights(case["ch"], seed))
        g1, g2, loss = 0, 0, 0.0
        for e in pairs_of(case, seed):
            e = E.field(e)
            r = E.tm(e, kappa, mu)
            h = E.layer(W1, r)
            d = E.layer(W2, h) - e
            loss += float(d.abs().square().sum())
            gh = E.layer_dag(W2, 2 * d)
            inner = lambda g, f: torch.stack([torch.stack([torch.stack([  # noqa: E731
                (g[..., a, :] * v[..., b, :].conj()).sum() for b in range(v.shape[-2])]) for a in range(g.shape[-2])])
                for v in (E.transport(f, k) for k in range(9))])
            g2 = g2 + inner(2 * d, h)
            g1 = g1 + inner(gh, r)
        return {"grad1": g1.cpu().numpy(), "grad2": g2.cpu().numpy(), "loss": np.float64(loss)}
    if kind == "net":
        W1, W2 = (_bf16(w) for w in weights(case["ch"], seed))
        fwd = lambda f: E.even(E.layer(W2, E.layer(W1, E.even(f))))          # noqa: E731
        adj = lambda f: E.even(E.layer_dag(W1, E.layer_dag(W2, E.even(f))))  # noqa: E731
        src = gaussian(L, n, seed)
        mid, out = torch.empty_like(src), torch.empty_like(src)
        for r in range(n):
            f = fwd(E.field(src[:, r]))
            mid[:, r], out[:, r] = f.reshape(V, 4, 3), adj(f).reshape(V, 4, 3)
        return [stored(mid, L, case["prec"], q.EVEN), stored(out, L, case["prec"], q.EVEN)]
    if kind == "operator":
        src, prec, sub = gaussian(L, n, seed), case["prec"], q.FULL
        op = lambda f: E.tm(f, kappa, mu)                                    # noqa: E731
        if case["form"] == "normal":
            sub = q.EVEN
            op = lambda f: E.normal(E.even(f), kappa, mu)                    # noqa: E731
    elif kind == "gauss":
        src, prec, sub = points(L, n, seed) if case["slice"] else gaussian(L, n, seed), "double", q.FULL

        def op(f):
            for _ in range(case["steps"]):
                f = (f + ALPHA_GAUSS * sum(E.transport(f, k) for k in range(1, 7))) / (1 + 6 * ALPHA_GAUSS)
            return f
    else:
        src, prec, sub = z2(L, 1, seed) if kind != "propagator" else points(L, n, seed), "double", q.FULL
        op = lambda f: E.solve(f, kappa, mu, kind == "cg")                   # noqa: E731
    out = torch.empty_like(src)
    for r in range(n):
        out[:, r] = op(E.field(src[:, r].contiguous())).reshape(V, 4, 3)
    return [stored(out, L, prec, sub)]
