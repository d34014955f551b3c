"""The work a user of gasoline_amd has it do, one case per kind of call.

A case names a kind of call and its sizes:

  gravity   new positions -> tree build -> gravity of every particle
  ensemble  the same over a batch of independent systems in one forest
  periodic  gravity in a periodic box with Ewald summation
  sph       search structure -> kNN + DenDVDX -> EOS -> SphPressureTermsSym
  step      one kick-drift-kick step, gravity and gas (evolve.KDK)
  block     one top step of block time steps, gravity and gas (BlockSteps)

prepare() holds what a simulation holds between steps: the handle with its
particle store on the GPU.  run() is one step of it.  Every handle call is
the public binding's; outputs come out with gg_get into tensors on the GPU.

FP32 and FP64 are the handle's two pair arithmetics.  Calls that are one
operator (gravity, ensemble, sph) come in both, the FP32 ones with an FP64
direct evaluation to be compared with; periodic boxes, whole steps and block
steps run in FP64.
"""
import ctypes
import math

import numpy as np
import torch

import gasoline_amd as gg
from gasoline_amd import evolve, ics

DEV = "cuda"
GAMMA = 5.0 / 3.0


def listed():
    return [
        # the smallest calls: a test problem or one small system, where the
        # launches and the host's waits are most of the time
        {"name": "gravity_4k_quad_f32", "kind": "gravity", "n": 4096, "prec": 32,
         "theta": 0.7, "order": 2},
        # a star cluster in the reference's precision at the accurate setting
        {"name": "gravity_30k_hexa_f64", "kind": "gravity", "n": 30011, "prec": 64,
         "theta": 0.55, "order": 4},
        # the accurate setting in FP32 at an ordinary size
        {"name": "gravity_300k_hexa_f32", "kind": "gravity", "n": 300007, "prec": 32,
         "theta": 0.55, "order": 4},
        # the reference's own configuration (theta 0.7, quadrupole) at a large size
        {"name": "gravity_2m_quad_f64", "kind": "gravity", "n": 2097152, "prec": 64,
         "theta": 0.7, "order": 2},
        # many small systems of uneven size at once
        {"name": "ensemble_48_hexa_f32", "kind": "ensemble", "nsys": 48, "nmin": 1024,
         "nmax": 16384, "prec": 32, "theta": 0.5, "order": 4},
        # a clustered periodic box with one replica shell and Ewald
        {"name": "periodic_200k_f64", "kind": "periodic", "n": 200000, "theta": 0.7,
         "nreps": 1},
        # a small gas box
        {"name": "sph_box_4k_f32", "kind": "sph", "n": 4096, "prec": 32, "K": 32,
         "shape": "box", "sorted": False},
        # a centrally concentrated gas sphere, open boundaries, arbitrary order
        {"name": "sph_sphere_100k_f32", "kind": "sph", "n": 100003, "prec": 32, "K": 64,
         "shape": "sphere", "sorted": False},
        # the adiabatic periodic box of the benchmark, in the reference's precision
        {"name": "sph_box_1m_f64", "kind": "sph", "n": 1048576, "prec": 64, "K": 64,
         "shape": "box", "sorted": True},
        # one step of a large gas collapse: everything the force path has
        {"name": "step_collapse_1.5m_f64", "kind": "step", "n": 1500001, "gas": 1.0, "K": 64,
         "theta": 0.55},
        # one step of a disk galaxy: gas a fifth of the particles
        {"name": "step_galaxy_250k_f64", "kind": "step", "n": 250000, "gas": 0.2, "K": 32,
         "theta": 0.55},
        # production stepping of a small galaxy: several force evaluations per
        # top step, most of them for a part of the particles
        {"name": "block_galaxy_50k_f64", "kind": "block", "n": 50000, "gas": 0.2, "K": 32,
         "theta": 0.7, "delta": 0.004},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gravity", "gravity", "ensemble", "periodic", "sph", "sph", "step",
                       "block"])
    if kind == "gravity":
        prec = rng.choice([32, 64])
        return {"kind": kind, "n": _loguniform(rng, 1000, 320000 if prec == 32 else 1600000),
                "prec": prec, "theta": rng.choice([0.5, 0.55, 0.6, 0.7, 0.8]),
                "order": rng.choice([2, 2, 3, 4, 4])}
    if kind == "ensemble":
        return {"kind": kind, "nsys": rng.randint(2, 64), "nmin": rng.choice([256, 1024]),
                "nmax": rng.choice([4096, 8192, 16384]), "prec": rng.choice([32, 64]),
                "theta": rng.choice([0.5, 0.6]), "order": rng.choice([2, 4])}
    if kind == "periodic":
        return {"kind": kind, "n": _loguniform(rng, 4000, 250000),
                "theta": rng.choice([0.6, 0.7]), "nreps": 1}
    if kind == "sph":
        prec = rng.choice([32, 64])
        return {"kind": kind, "n": _loguniform(rng, 2000, 110000 if prec == 32 else 1000000),
                "prec": prec, "K": rng.choice([32, 48, 64]),
                "shape": rng.choice(["box", "sphere"]), "sorted": rng.random() < 0.5}
    if kind == "step":
        return {"kind": kind, "n": _loguniform(rng, 8000, 1000000),
                "gas": rng.choice([1.0, 0.5, 0.2]), "K": rng.choice([32, 64]),
                "theta": rng.choice([0.55, 0.7])}
    return {"kind": kind, "n": _loguniform(rng, 6000, 100000), "gas": rng.choice([0.2, 0.5]),
            "K": 32, "theta": rng.choice([0.55, 0.7]), "delta": 0.004}


# ------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _f32(x):
    """Positions as a particle file stores them: FP32 values held in FP64."""
    return x.float().double().contiguous()


def _iso(g, n):
    z, ph = 2 * _uniform(g, n) - 1, 2 * math.pi * _uniform(g, n)
    s = torch.sqrt(1 - z * z)
    return torch.stack([s * torch.cos(ph), s * torch.sin(ph), z], 1)


def _plummer(g, n):
    """Plummer sphere, G = M = a = 1, cut at 99.9 per cent of the mass."""
    x = torch.clamp(0.999 * _uniform(g, n), min=1e-10)
    return _f32(_iso(g, n) / torch.sqrt(x ** (-2.0 / 3.0) - 1)[:, None])


def _clustered_box(g, n):
    """Half uniform, half in three clumps, in [-1/2, 1/2)^3."""
    u = _uniform(g, n // 2, 3) - 0.5
    c = _uniform(g, 3, 3) - 0.5
    k = (3 * _uniform(g, n - n // 2)).long().clamp(max=2)
    cl = c[k] + 0.03 * _normal(g, n - n // 2, 3)
    return _f32((torch.cat([u, cl]) + 0.5) % 1.0 - 0.5)


def _curve_order(r):
    """Order along a space-filling curve, as a store that is kept sorted has it."""
    lo = r.min(0).values
    q = ((r - lo) / (r.max() - r.min() + 1e-300) * 1023).long().clamp(0, 1023)
    key = torch.zeros(len(r), dtype=torch.long, device=r.device)
    for b in range(10):
        for d in range(3):
            key |= ((q[:, d] >> b) & 1) << (3 * b + d)
    return torch.argsort(key, stable=True)


def _gas(case, seed):
    """Gas of an sph case: r, v, u, m and the period (None: open)."""
    g, n = _gen(seed), case["n"]
    if case["shape"] == "box":
        # a 2^-24 lattice in [0, 1)^3, velocities sigma 0.1, u = 1
        r = torch.randint(0, 1 << 24, (n, 3), generator=g, device=DEV).double() / (1 << 24)
        v, u, period = _f32(0.1 * _normal(g, n, 3)), 1.0, [1.0, 1.0, 1.0]
    else:
        # density ~ 1/r inside R = 1, falling in, u = 0.05
        r = _f32(_iso(g, n) * torch.sqrt(_uniform(g, n))[:, None])
        v, u, period = _f32(-0.5 * r + 0.05 * _normal(g, n, 3)), 0.05, None
    if case["sorted"]:
        o = _curve_order(r)
        r, v = r[o].contiguous(), v[o].contiguous()
    return r, v, torch.full((n,), u, dtype=torch.float64, device=DEV), \
        torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV), period


def _systems(case):
    """Offsets of the ensemble's systems, their sizes log-uniform; the same
    for every seed (an ensemble keeps its systems while they move)."""
    u = torch.rand(case["nsys"], generator=torch.Generator().manual_seed(case["nsys"]),
                   dtype=torch.float64)
    ns = torch.exp(math.log(case["nmin"]) + u * math.log(case["nmax"] / case["nmin"])).long()
    return [0] + torch.cumsum(ns, 0).tolist()


GRAV_SOFT = 0.01       # softening of the isolated spheres
ENS_SOFT = 0.005


def _grav_inputs(case, seed):
    """r, m, softening and, for an ensemble, the systems' offsets."""
    g, kind = _gen(seed), case["kind"]
    if kind == "gravity":
        n = case["n"]
        return _plummer(g, n), torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV), \
            GRAV_SOFT, None
    if kind == "periodic":
        n = case["n"]
        return _clustered_box(g, n), torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV), \
            0.2 / n ** (1 / 3), None
    off = _systems(case)
    m = torch.cat([torch.full((b - a,), 1.0 / (b - a), dtype=torch.float64, device=DEV)
                   for a, b in zip(off[:-1], off[1:])])
    return _plummer(g, off[-1]), m, ENS_SOFT, off


def _galaxy(case, seed):
    """Gas and collisionless particles of a step or block case."""
    n = case["n"]
    if case["gas"] == 1.0:
        g = _gen(seed)
        r = _f32(_iso(g, n) * torch.sqrt(_uniform(g, n))[:, None])
        o = _curve_order(r)
        r = r[o].contiguous()
        return dict(r=r, v=_f32(-0.3 * r + 0.02 * _normal(g, n, 3)),
                    m=torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV),
                    u=torch.full((n,), 0.05, dtype=torch.float64, device=DEV),
                    soft=torch.full((n,), 0.004, dtype=torch.float64, device=DEV),
                    gas=torch.ones(n, dtype=torch.bool, device=DEV))
    ng = int(round(n * case["gas"]))
    d = ics.disk_galaxy(n - ng, ng, seed=int(seed) % (1 << 31))
    return {k: torch.as_tensor(d[k], device=DEV) for k in ("r", "v", "m", "u", "soft", "gas")}


# ------------------------------------------------------------ prepare
def _buffers(names, n):
    out = {}
    for name in names:
        w = gg.FIELDS[name][1]
        kind = torch.int32 if name == "iRung" else torch.float64
        out[name] = torch.empty((n, w) if w > 1 else (n,), dtype=kind, device=DEV)
    return out


def _fetch(pk, out):
    """The named fields of the store into tensors on the GPU."""
    for name, t in out.items():
        rc = gg.lib().gg_get(pk.h, gg.FIELDS[name][0], ctypes.c_void_p(t.data_ptr()), 1)
        if rc:
            raise gg.GGError(gg.lib().gg_last_error().decode(errors="replace"))
    return out


def _prec(case):
    return gg.PREC_FP32 if case.get("prec") == 32 else gg.PREC_FP64


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("gravity", "ensemble", "periodic"):
        s["r"], m, soft, s["off"] = _grav_inputs(case, seed)
        n = len(m)
        pk = s["pk"] = gg.Pkd(n, prec=_prec(case))
        pk.put("r", s["r"])
        pk.put("fMass", m)
        pk.put("fSoft", torch.full_like(m, soft))
        if s["off"] is not None:
            s["off"] = np.asarray(s["off"], np.int32)
        if kind == "periodic":
            pk.set_period([1.0, 1.0, 1.0])
        # the timestep criterion's dtGrav is taken in the reference's precision
        s["out"] = _buffers(("a", "fPot") + (("dtGrav",) if _prec(case) == gg.PREC_FP64 else ()),
                            n)
        return s
    if kind == "sph":
        s["r"], v, u, m, s["period"] = _gas(case, seed)
        n = len(m)
        pk = s["pk"] = gg.Pkd(n, prec=_prec(case))
        pk.put("r", s["r"])
        pk.put("vPred", v)
        pk.put("uPred", u)
        pk.put("fMass", m)
        s["zero"] = torch.zeros_like(u)
        s["smf"] = gg.Smf.default()
        s["out"] = _buffers(("fBall2", "fDensity", "divv", "curlv", "a", "uDotPdV", "uDotAV"), n)
        return s
    d = _galaxy(case, seed)
    n = len(d["m"])
    s["d"] = d
    pk = s["pk"] = gg.Pkd(n, prec=gg.PREC_FP64)
    for name, key in (("r", "r"), ("v", "v"), ("vPred", "v"), ("fMass", "m"), ("fSoft", "soft"),
                      ("u", "u"), ("uPred", "u")):
        pk.put(name, d[key])
    on = gg.TYPE_ACTIVE | gg.TYPE_TREEACTIVE
    bits = torch.where(d["gas"], on | gg.TYPE_SMOOTHACTIVE | gg.TYPE_GAS, on | gg.TYPE_DARK)
    pk.put("iActive", bits.int())
    smf = gg.Smf.default(iViscosityLimiter=1)
    if kind == "step":
        s["dt"] = 1e-3 if case["gas"] == 1.0 else 5e-4
        s["run"] = evolve.KDK(pk, smf, nSmooth=case["K"], theta=case["theta"], iOrder=4)
        s["run"].forces(s["dt"])
        s["out"] = _buffers(("r", "v", "u", "a", "fDensity"), n)
    else:
        s["rung0"] = torch.zeros(n, dtype=torch.int32, device=DEV)
        s["run"] = gg.BlockSteps(pk, case["delta"], iMaxRung=5, smf=smf, dTheta=case["theta"],
                                 iOrder=4, nSmooth=case["K"])
        s["run"].forces(0)
        s["out"] = _buffers(("r", "v", "u", "a", "fDensity", "iRung"), n)
    return s


# ---------------------------------------------------------------- run
def run(s):
    case, pk = s["case"], s["pk"]
    kind = case["kind"]
    if kind in ("gravity", "ensemble", "periodic"):
        pk.put("r", s["r"])
        order = case.get("order", 4)
        if kind == "ensemble":
            pk.build_forest(s["off"], 16, 1, case["theta"], order)
        else:
            pk.build_binary(16, 1, case["theta"], order)
        pk.init_accel()
        if kind == "periodic":
            st = pk.grav_all(order, nReps=case["nreps"], periodic=True, bEwald=True)
        else:
            st = pk.grav_all(order)
        return dict(_fetch(pk, s["out"]), stats=st)
    if kind == "sph":
        per, K, smf = s["period"] is not None, case["K"], s["smf"]
        pk.put("r", s["r"])
        pk.put("fBall2", s["zero"])         # no search radius from before
        pk.init_accel()
        pk.build_local(period=s["period"])
        pk.smooth(smf, K, per)
        pk.gas_pressure(smf)
        pk.resmooth(smf, K, per)
        return _fetch(pk, s["out"])
    d = s["d"]                              # back to the start of the step
    for name, key in (("r", "r"), ("v", "v"), ("vPred", "v"), ("u", "u"), ("uPred", "u")):
        pk.put(name, d[key])
    if kind == "step":
        s["run"].step(s["dt"])
    else:
        pk.put("iRung", s["rung0"])
        s["run"].s.iCurrMaxRung = 0
        s["run"].top_step()
    return _fetch(pk, s["out"])


# --------------------------------------------------------------- work
def work(case):
    """Each input read once, each output written once, and the arithmetic of
    the interactions themselves (38 operations a particle pair, 76 to 312 a
    cell, about 90 a density pair and 220 a force pair), with list lengths of
    an ordinary particle."""
    kind = case["kind"]

    def gravity(n, theta, order, reps=1):
        cells = 130.0 * math.log2(max(n / 256.0, 2.0)) / 12.0 * (0.7 / theta) ** 3
        flop = {1: 45, 2: 76, 3: 155, 4: 312}[order]
        return n * (24 + 16 + 40), n * (cells * flop + 150 * 38) * reps

    def sph(n, K):
        return n * (24 + 24 + 16 + 112), n * K * (90 + 220)

    if kind == "gravity":
        b, f = gravity(case["n"], case["theta"], case["order"])
    elif kind == "ensemble":
        mean = (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        b, f = gravity(mean, case["theta"], case["order"])
        b, f = b * case["nsys"], f * case["nsys"]
    elif kind == "periodic":
        b, f = gravity(case["n"], case["theta"], 4, 1.5)
        f += case["n"] * (80 * 447 + 92 * 58)
    elif kind == "sph":
        b, f = sph(case["n"], case["K"])
    else:
        b, f = gravity(case["n"], case["theta"], 4)
        b2, f2 = sph(case["n"] * case["gas"], case["K"])
        b, f = b + b2 + 200 * case["n"], f + f2
        if kind == "block":
            b, f = 4 * b, 4 * f
    return {"bytes": b, "flops": f}


# -------------------------------------------------------------- exact
def exact(case, seed):
    """The FP32 calls in 64 bits without a tree: gravity by direct sum, the
    gas by a full search for each particle's neighbours.  The other cases
    compute in FP64 themselves."""
    if case.get("prec") != 32:
        return None
    if case["kind"] == "sph":
        return _exact_sph(case, seed)
    r, m, soft, off = _grav_inputs(case, seed)
    a, pot = torch.empty_like(r), torch.empty_like(m)
    off = off or [0, len(m)]
    for lo, hi in zip(off[:-1], off[1:]):
        a[lo:hi], pot[lo:hi] = _direct(r[lo:hi], m[lo:hi], 2 * soft)
    return {"a": a, "fPot": pot, "stats": None}


def _direct(r, m, twoh):
    """Accelerations and potentials of one system, spline-softened inside
    twoh (Hernquist & Katz 1989), every pair."""
    n = len(m)
    rows = max(1, min(n, (1 << 25) // n))
    acc, pot = torch.empty_like(r), torch.empty_like(m)
    src = torch.cat([r, torch.ones(n, 1, dtype=r.dtype, device=r.device)], 1) * m[:, None]
    dih = 2.0 / twoh
    for lo in range(0, n, rows):
        x = r[lo:lo + rows]
        d2 = (x[:, None, 0] - r[None, :, 0]).square_()
        for d in (1, 2):
            d2 += (x[:, None, d] - r[None, :, d]).square_()
        i, j = torch.nonzero(d2 < twoh * twoh, as_tuple=True)
        u = torch.sqrt(d2[i, j]) * dih
        phi = d2.rsqrt_()
        ui = torch.clamp(u, min=1e-300)
        pin = dih * (7 / 5 - 2 / 3 * u ** 2 + 3 / 10 * u ** 4 - u ** 5 / 10)
        pout = dih * (-1 / (15 * ui) + 8 / 5 - 4 / 3 * u ** 2 + u ** 3 - 3 / 10 * u ** 4
                      + u ** 5 / 30)
        fin = dih ** 3 * (4 / 3 - 6 / 5 * u ** 2 + u ** 3 / 2)
        fout = dih ** 3 * (-1 / (15 * ui ** 3) + 8 / 3 - 3 * u + 6 / 5 * u ** 2 - u ** 3 / 6)
        other = (i + lo != j).to(r.dtype)
        phi[i, j] = torch.where(u < 1, pin, pout) * other
        pot[lo:lo + rows] = -(phi @ m)
        phi.pow_(3)
        phi[i, j] = torch.where(u < 1, fin, fout) * other
        w = phi @ src
        acc[lo:lo + rows] = w[:, :3] - x * w[:, 3:]
    return acc, pot


def _image(d, period):
    return d if period is None else d - torch.round(d)


def _w(q):
    """M4 kernel without its normalisation, q = r / h (2h the support)."""
    t = 2 - q
    return torch.where(q < 1, 1 - 0.75 * t * q * q, 0.25 * t ** 3)


def _dw(q):
    return torch.where(q < 1, -3 + 2.25 * q, -0.75 * (2 - q) ** 2 / torch.clamp(q, min=1e-300))


def _exact_sph(case, seed):
    r, v, u, m, period = _gas(case, seed)
    n, K = len(m), case["K"]
    nb = torch.empty(n, K, dtype=torch.long, device=DEV)
    d2 = torch.empty(n, K, dtype=torch.float64, device=DEV)
    rows = max(1, min(n, (1 << 25) // n))
    for lo in range(0, n, rows):
        s = _image(r[lo:lo + rows, None, 0] - r[None, :, 0], period).square_()
        for d in (1, 2):
            s += _image(r[lo:lo + rows, None, d] - r[None, :, d], period).square_()
        d2[lo:lo + rows], nb[lo:lo + rows] = torch.topk(s, K, dim=1, largest=False)
    ball = d2.max(1).values
    ih2 = 4 / ball
    q = torch.sqrt(d2 * ih2[:, None])
    dx = _image(r[:, None] - r[nb], period)                     # p - q
    dv = v[:, None] - v[nb]
    mq = m[nb]
    rho = (_w(q) * mq).sum(1) * ih2 ** 1.5 / math.pi
    rs = _dw(q) * mq
    G = -torch.einsum("nk,nka,nkb->nab", rs, dv, dx)            # sum (v_q - v_p)_a dx_b rs
    f = 3 / (d2 * rs).sum(1).abs()
    divv = f * (G[:, 0, 0] + G[:, 1, 1] + G[:, 2, 2])
    curl = f[:, None] * torch.stack([G[:, 2, 1] - G[:, 1, 2], G[:, 0, 2] - G[:, 2, 0],
                                     G[:, 1, 0] - G[:, 0, 1]], 1)
    pr2, c = (GAMMA - 1) * u / rho, torch.sqrt(GAMMA * (GAMMA - 1) * u)
    # each pair as list owner p meets it, both ends
    rs1 = _dw(q) * (0.5 / math.pi * ih2 ** 2 / torch.sqrt(0.25 * ball))[:, None]
    vr = (dv * dx).sum(2)
    mu = torch.where(vr < 0, -vr / torch.sqrt(torch.clamp(d2, min=1e-300)),
                     torch.zeros_like(vr))
    visc = ((c[:, None] + c[nb]) + 2.0 * 1.5 * mu) * mu / (rho[:, None] + rho[nb])
    both = pr2[:, None] + pr2[nb] + visc
    mp = m[:, None]
    idx = nb.reshape(-1)
    acc = -((both * rs1 * mq)[:, :, None] * dx).sum(1)
    acc.index_add_(0, idx, ((both * rs1 * mp)[:, :, None] * dx).reshape(-1, 3))
    pdv = (rs1 * mq * pr2[:, None] * vr).sum(1)
    pdv.index_add_(0, idx, (rs1 * mp * pr2[nb] * vr).reshape(-1))
    av = (rs1 * mq * 0.5 * visc * vr).sum(1)
    av.index_add_(0, idx, (rs1 * mp * 0.5 * visc * vr).reshape(-1))
    return {"fBall2": ball, "fDensity": rho, "divv": divv, "curlv": curl, "a": acc,
            "uDotPdV": pdv, "uDotAV": av}
