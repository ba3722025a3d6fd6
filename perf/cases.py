"""What the framework is timed on, through its public entry points
(ifos3d-dev_amd/ifosgpu.py): one time step, whole gradient shots and batches,
forward solves, the two time-domain gradients, the frequency-domain gradient
and Hessian, and the optimiser's part of an inversion iteration.

`listed()` names the cases, `draw()` gives more of the same ranges,
`prepare()` makes what a caller holds before the call (inputs from the seed,
the context or history it keeps), `run()` is one pass, `work()` the bytes and
operations a pass cannot do without, and `exact()` the pass in 64 bits from
the scheme's equations alone (torch, no code of this repository).

Shapes are those of the workloads in ifos3d-dev_amd/workloads.py (84^3,
276^3, 404 x 212 x 404 halved, 536 x 280 x 536, the three grid levels), with
fewer time steps; the wavelet is shifted and the receivers stand close enough
to the source that the signal arrives within the record.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ifos3d-dev_amd"))
import ifosgpu as ig  # noqa: E402

DEV = "cuda"
VMAX = 5500.0
GAMMA4 = 1.184614  # the CFL factor of the 4th-order Holberg operators


# ---------------------------------------------------------------------------
# the cases
def listed():
    return [
        # one time step of a caller with its own loop (the reference's call order), small grid
        dict(name="step_84", path="step", nx=84, ny=84, nz=84, fw=10, dh=2.0, L=0, nf=3, kahan=False, fs=0, ntr=32),
        # a whole gradient shot of the toy inversion: launch-bound
        dict(name="shot_84", path="shot", nx=84, ny=84, nz=84, fw=10, dh=2.0, nt=600, L=0, nf=3, kahan=False, fs=0,
             ntr=32, src=1),
        # the benchmark's grid, one shot through the one-shot context
        dict(name="shot_276", path="shot", nx=276, ny=276, nz=276, fw=10, dh=4.0, nt=100, L=0, nf=6, kahan=False,
             fs=0, ntr=1024, src=1),
        # the viscoelastic case: three mechanisms, compensated DFT sums, eight frequencies
        dict(name="shot_visco", path="shot", nx=202, ny=106, nz=202, fw=10, dh=5.0, nt=100, L=3, nf=8, kahan=True,
             fs=0, ntr=1024, src=1),
        # a batch of the toy inversion's four shots, replayed as a graph, compensated sums
        dict(name="batch_84", path="batch", nx=84, ny=84, nz=84, fw=10, dh=2.0, nt=300, L=0, nf=3, kahan=True, fs=0,
             ntr=32, src=1, shots=4, adjoint=True, graph=True),
        # the benchmark's grid, a batch of gradient shots
        dict(name="batch_276", path="batch", nx=276, ny=276, nz=276, fw=10, dh=4.0, nt=60, L=0, nf=6, kahan=False,
             fs=0, ntr=1024, src=1, shots=4, adjoint=True, graph=False),
        # the largest grid: forward modelling of one shot, 64 x 64 receivers
        dict(name="forward_536", path="batch", nx=536, ny=280, nz=536, fw=12, dh=5.0, nt=40, L=0, nf=1, kahan=False,
             fs=0, ntr=4096, src=1, shots=1, adjoint=False, graph=False),
        # forward solves of three uneven grid levels together
        dict(name="levels", path="levels", n0=116, n1=148, n2=212, fw=10, dh=4.0, nt=64, shots=3, ntr=64),
        # the full-band time-domain gradient of one shot
        dict(name="timegrad_148", path="td", nx=148, ny=148, nz=148, fw=10, dh=4.0, nt=64, L=0, fs=0, ntr=256, src=1),
        # the exact discrete adjoint of one shot
        dict(name="adjoint_116", path="adj", nx=116, ny=116, nz=116, fw=10, dh=4.0, nt=64, ntr=256),
        # the frequency-domain gradient and the diagonal Hessian from stored DFT fields
        dict(name="gradhess_276", path="hess", nx=276, ny=276, nz=276, fw=10, dh=4.0, nf=6),
        # the optimiser between two gradients: taper, L-BFGS direction, test model
        dict(name="update_276", path="update", nx=276, ny=276, nz=276, fw=10, dh=4.0, method="lbfgs", damp=2, nsrc=16,
             ntr=1024),
    ]


def draw(rng):
    path = rng.choice(["step", "shot", "shot", "batch", "batch", "levels", "td", "adj", "hess", "update"])

    def sizes(lo, hi, most):
        while True:
            n = [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) for _ in range(3)]
            if n[0] * n[1] * n[2] <= most:
                return dict(zip(("nx", "ny", "nz"), n))

    fw = rng.choice([6, 8, 10, 10, 12])
    dh = rng.choice([2.0, 4.0, 5.0, 3.0])
    ntr = int(round(math.exp(rng.uniform(math.log(16), math.log(2048)))))
    if path == "step":
        return dict(path=path, **sizes(40, 300, 20e6), fw=fw, dh=dh, L=rng.choice([0, 0, 1, 3]),
                    nf=rng.randint(1, 8), kahan=rng.random() < 0.3, fs=rng.choice([0, 0, 1]), ntr=ntr)
    if path == "shot":
        g = sizes(40, 280, 18e6)
        nt = max(30, min(400, int(6e8 / (g["nx"] * g["ny"] * g["nz"]))))
        return dict(path=path, **g, fw=fw, dh=dh, nt=rng.randint(nt // 2, nt), L=rng.choice([0, 0, 0, 1, 3]),
                    nf=rng.randint(1, 8), kahan=rng.random() < 0.3, fs=rng.choice([0, 0, 0, 1]), ntr=ntr,
                    src=rng.choice([1, 1, 2, 3, 4]))
    if path == "batch":
        g = sizes(40, 280, 18e6)
        shots = rng.randint(1, 4)
        nt = max(20, min(300, int(6e8 / (shots * g["nx"] * g["ny"] * g["nz"]))))
        return dict(path=path, **g, fw=fw, dh=dh, nt=rng.randint(nt // 2, nt), L=rng.choice([0, 0, 0, 1, 3]),
                    nf=rng.randint(1, 8), kahan=rng.random() < 0.3, fs=rng.choice([0, 0, 0, 1]), ntr=ntr,
                    src=rng.choice([1, 1, 2, 3, 4]), shots=shots, adjoint=rng.random() < 0.7,
                    graph=rng.random() < 0.4)
    if path == "levels":
        n = sorted(rng.randint(60, 212) for _ in range(3))
        return dict(path=path, n0=n[0], n1=n[1], n2=n[2], fw=10, dh=dh, nt=rng.randint(30, 64),
                    shots=rng.randint(1, 3), ntr=rng.randint(16, 256))
    if path == "td":
        return dict(path=path, **sizes(48, 200, 3.2e6), fw=fw, dh=dh, nt=rng.randint(30, 64),
                    L=rng.choice([0, 0, 1]), fs=rng.choice([0, 0, 1]), ntr=ntr, src=rng.choice([1, 1, 2]))
    if path == "adj":
        return dict(path=path, **sizes(48, 150, 1.5e6), fw=fw, dh=dh, nt=rng.randint(30, 64), ntr=min(ntr, 400))
    if path == "hess":
        return dict(path=path, **sizes(64, 300, 20e6), fw=fw, dh=dh, nf=rng.randint(1, 8))
    return dict(path=path, **sizes(64, 300, 20e6), fw=fw, dh=dh, method=rng.choice(["lbfgs", "cg"]),
                damp=rng.choice([0, 1, 2]), nsrc=rng.randint(1, 24), ntr=ntr)


# ---------------------------------------------------------------------------
# inputs
class _Rand:
    """seeded random fields on the device"""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)
        self.np = np.random.default_rng(seed)

    def smooth(self, shape, cells=10):
        """values of about [-1, 1], varying over `cells` cells"""
        coarse = [max(2, -(-s // cells) + 1) for s in shape]
        a = torch.rand(coarse, generator=self.gen, device=DEV) * 2.0 - 1.0
        return torch.nn.functional.interpolate(a[None, None], size=shape, mode="trilinear", align_corners=True)[0, 0]


def _dev(a, G):
    """a canonical array (ny+5, nx+5, nz+5) in the device layout"""
    out = torch.zeros(G.dshape, device=DEV)
    out[..., ig.KOFF - 2:ig.KOFF - 2 + G.nz + 5] = a
    return out


def _dt(c):
    return float(np.float32(0.9 * c["dh"] / (GAMMA4 * math.sqrt(3.0) * VMAX)))


def _inputs(c, seed):
    """what a shot case's numbers are made from, on the grid of `c`: the
    model (canonical float arrays), source, receivers and wavelet; no
    library object"""
    r = _Rand(seed)
    shape = (c["ny"] + 5, c["nx"] + 5, c["nz"] + 5)
    vp = 4000.0 + 1000.0 * r.smooth(shape, 20)
    vs = vp / (1.85 + 0.15 * r.smooth(shape, 20))
    rho = 310.0 * vp ** 0.25
    m = dict(rho=rho, pi=rho * vp * vp, u=rho * vs * vs)
    if c.get("L"):
        # Q of 20-100 per cell, mechanisms spread over 5-40 Hz
        q = 60.0 + 40.0 * r.smooth(shape, 6)
        m["taus"] = (2.0 / q).contiguous()
        m["taup"] = (1.6 / q).contiguous()
        fl = np.geomspace(4.0, 50.0, c["L"] + 1)[:c["L"]]
        # unrelaxed moduli stay below VMAX: L * tau <= 0.3
        m["eta"] = [float(np.float32(_dt(c) * 2.0 * math.pi * f)) for f in fl]
        m["pi"] = m["pi"] / (1.0 + c["L"] * m["taup"])
        m["u"] = m["u"] / (1.0 + c["L"] * m["taus"])
    return r, m


def _shot(c, r, nt):
    """a source in the interior and receivers around it, and the record's
    observed traces: direct arrivals of the same wavelet with noise"""
    fw, dt = c["fw"], _dt(c)
    n = (c["nx"], c["ny"], c["nz"])
    T = nt * dt
    fc = float(np.float32(max(1.0 / (0.6 * T), 5.0)))
    # the middle third of the interior
    s = [int(r.np.integers(fw + 1 + (q - 2 * fw) // 3, fw + 2 + (2 * (q - 2 * fw)) // 3)) for q in n]
    reach = max(4, int(0.35 * 4000.0 * T / c["dh"]))
    rec = np.stack([np.clip(s[a] + r.np.integers(-reach, reach + 1, c["ntr"]), fw + 1, n[a] - fw)
                    for a in range(3)], 1).astype(np.int32)
    src = (s[0], s[1], s[2], float(np.float32(-1.0 / fc)), fc, 1.0, c.get("src", 1))
    dist = np.linalg.norm((rec - np.array(s)) * c["dh"], axis=1)
    t = (np.arange(nt + 1) * dt)[None, None, :]
    tau = math.pi * fc * (t - 0.5 / fc - dist[None, :, None] / 4000.0)
    amp = r.np.uniform(-1.0, 1.0, (3, c["ntr"], 1)) / (dist[None, :, None] + c["dh"])
    # about the size of a unit source's velocities
    scale = dt / (2000.0 * c["dh"] ** 3) * (1.0 if c.get("src", 1) == 1 else 2000.0 * 2000.0)
    obs = scale * (amp * (1 - 2 * tau * tau) * np.exp(-tau * tau) + 0.02 * r.np.standard_normal(tau.shape))
    obs[..., 0] = 0.0
    return src, rec, obs.astype(np.float32)


def _finv(c, nt):
    """DFT frequencies around the wavelet's band"""
    fc = max(1.0 / (0.6 * nt * _dt(c)), 5.0)
    return [float(np.float32(f)) for f in np.linspace(0.4, 1.4, c["nf"]) * fc]


TAST = 100
VPPML = 4500.0


def _geom(c, nt):
    return ig.Geom(c["nx"], c["ny"], c["nz"], c["fw"], c["dh"], c["dh"], c["dh"], _dt(c), nt, 2, c.get("fs", 0))


def _fpml(c, nt):
    return float(np.float32(max(1.0 / (0.6 * nt * _dt(c)), 5.0)))


def _level_cases(c):
    """the three levels of one cube: the spacing grows as the cells get fewer"""
    out = []
    for n in (c["n0"], c["n1"], c["n2"]):
        dh = float(np.float32(c["dh"] * (c["n2"] - 2 * c["fw"]) / (n - 2 * c["fw"])))
        out.append(dict(nx=n, ny=n, nz=n, fw=c["fw"], dh=dh, nt=max(20, int(round(c["nt"] * c["dh"] / dh))),
                        ntr=c["ntr"], L=0, nf=1, fs=0, src=1))
    return out


# ---------------------------------------------------------------------------
# what a caller holds before the call
def _context(cls, c, m, G, nt, *args):
    """a ShotContext or BatchContext of the case with its model set"""
    prec = ig.DFT_KAHAN if c.get("kahan") else ig.DFT_COMPAT
    k = cls(G, *args, prec) if cls is ig.ShotContext else cls(G, *args, prec, chunk=16)
    torch.cuda.synchronize()
    k.set_model(*[_dev(m[n], G) for n in ("rho", "pi", "u")])
    if c.get("L"):
        k.set_visco(_dev(m["taus"], G), _dev(m["taup"], G), m["eta"])
    k.set_cpml(VPPML, _fpml(c, nt))
    k.set_freqs(_finv(c, nt) if "nf" in c else [20.0], TAST)
    torch.cuda.synchronize()
    return k


def _prepare_step(c, seed):
    r, m = _inputs(c, seed)
    G = _geom(c, 200)
    s = dict(c=c, G=G, f=[_dev(_field(r, c, n), G) for n in range(9)])
    model = [_dev(m[n], G) for n in ("rho", "pi", "u")]
    for a in model:
        ig.matcopy_wrap(G, a)
    av = [torch.zeros(G.dshape, device=DEV) for _ in range(6)]
    ig.av_mat(G, model[0], model[2], av)
    s["m"] = model + av
    s["prof"] = torch.from_numpy(ig.cpml_profiles(G, VPPML, _fpml(c, 200))).to(DEV)
    s["ps"], s["pv"] = [[torch.zeros(G.psi_shape(n), device=DEV) for n in range(9)] for _ in range(2)]
    s["L"] = c["L"]
    if c["L"]:
        tau = [_dev(m[n], G) for n in ("taus", "taup")]
        for a in tau:
            ig.matcopy_wrap(G, a)
        tav = [torch.zeros(G.dshape, device=DEV) for _ in range(3)]
        ig.av_tau(G, tau[0], tav)
        s["r"] = [torch.zeros((c["L"],) + G.dshape, device=DEV) for _ in range(6)]
        s["tau"] = tau + tav
        s["visco"] = ig.visco_struct(s["r"], *tau, *tav, m["eta"])
    src, rec, _ = _shot(c, r, 200)
    s["sig"] = torch.from_numpy(ig.wavelet(G, 1, src[3], src[4], src[5])).to(DEV)
    s["src"] = torch.tensor([[src[0], src[1], src[2], 1]], dtype=torch.int32, device=DEV)
    s["rec"] = torch.from_numpy(rec).to(DEV)
    s["sec"] = torch.zeros((3, c["ntr"], 201), device=DEV)
    s["F"] = [torch.zeros((c["nf"],) + G.dshape, device=DEV) for _ in range(6)]
    s["C"] = [torch.zeros((c["nf"],) + G.dshape, device=DEV) for _ in range(6)] if c["kahan"] else None
    s["finv"] = _finv(c, 200)
    return s


def _field(r, c, n):
    """a wavefield of about 1e-3 m/s and the stress that goes with it, zero outside the grid"""
    a = torch.zeros((c["ny"] + 5, c["nx"] + 5, c["nz"] + 5), device=DEV)
    a[3:-2, 3:-2, 3:-2] = r.smooth((c["ny"], c["nx"], c["nz"]), 6) * (1e-3 if n < 3 else 8e3)
    return a


def _prepare_hess(c, seed):
    r = _Rand(seed)
    _, m = _inputs(c, seed)
    G = _geom(c, 100)
    F, B = [], []
    for n in range(6):
        for out, slots in ((F, c["nf"]), (B, 2 * c["nf"])):
            a = torch.zeros((slots,) + G.dshape, device=DEV)
            base = r.smooth((c["ny"], c["nx"], c["nz"]), 8) * 1e-6
            for l in range(slots):  # another frequency: shifted and scaled
                a[l, 3:-2, 3:-2, ig.KOFF + 1:ig.KOFF + 1 + c["nz"]] = torch.roll(
                    base, (3 * l + n, 5 * l, 7 * l + 1), (0, 1, 2)) * (1.0 - 0.07 * l)
            out.append(a)
    model = [_dev(m[n], G) for n in ("rho", "pi", "u")]
    out = [torch.zeros(G.dshape, device=DEV) for _ in range(6)]
    return dict(c=c, G=G, F=F, B=B, m=model + [None] * 6, out=out, finv=_finv(c, 100))


def _update_inputs(c, seed):
    """gradients g_1..g_5 of the last iterations (vp, vs; the last with rho),
    steps s_1..s_4 with positive curvature, the model and the taper points"""
    r, m = _inputs(c, seed)
    shape = (c["ny"], c["nx"], c["nz"])

    def field():
        return r.smooth(shape, 12) + 0.05 * r.smooth(shape, 4)

    g = [torch.stack([field() for _ in range(3)])]
    y, s = [], []
    for n in range(4):
        d = 0.3 * torch.stack([field() for _ in range(3)])
        y.append(d)
        g.append(g[-1] - d)
    for n in range(4):
        step = 0.01 * (1.0 + 0.2 * n) * y[n][:2]
        s.append((step - (0.005 * g[4][:2] if n == 3 else 0.0)).contiguous())
    rng = r.np
    n = (c["nx"], c["ny"], c["nz"])
    src = np.stack([rng.integers(c["fw"] + 1, q - c["fw"] + 1, c["nsrc"]) for q in n], 1)
    rec = np.stack([rng.integers(c["fw"] + 1, q - c["fw"] + 1, c["ntr"]) for q in n], 1)
    rec[:, 1] = c["fw"] + 1  # a plane of receivers under the top
    return m, g, s, src.astype(np.int32), rec.astype(np.int32)


def _prepare_update(c, seed):
    m, g, s, src, rec = _update_inputs(c, seed)
    G = _geom(c, 100)

    def dev(a):
        out = torch.zeros(G.dshape, device=DEV)
        out[3:-2, 3:-2, ig.KOFF + 1:ig.KOFF + 1 + c["nz"]] = a
        return out

    st = dict(c=c, G=G, src=src, rec=rec, n=G.field_elems())
    st["m"] = [_dev(m[n], G) for n in ("rho", "pi", "u")]
    st["test"] = [torch.zeros(G.dshape, device=DEV) for _ in range(3)]
    st["grad"] = [dev(a) for a in g[4]]
    st["work"] = [torch.zeros(G.dshape, device=DEV) for _ in range(3)]

    def tapered(a):
        t = [dev(x) for x in a]
        torch.cuda.synchronize()
        ig.precon_grad(G, t, c["damp"], src, rec)
        return t

    if c["method"] == "lbfgs":
        lb = ig.Lbfgs(G, numpar=2, bfgsnum=5)
        t = tapered(g[0])
        lb.savegrad(t[0], t[1])
        for it in (2, 3, 4, 5):
            torch.cuda.synchronize()
            lb.mod(it - 1).copy_from(ig.DBuf.wrap(s[it - 2].data_ptr(), (lb.n,)))
            if it < 5:
                t = tapered(g[it - 1])
                lb.update(t[0], t[1], it)
        st["lb"], st["slot"] = lb, lb.mod(5)
    else:
        st["prior"] = tapered(g[3]) + tapered(g[3])
    torch.cuda.synchronize()
    return st


def prepare(case, seed):
    c = dict(case)
    path = c["path"]
    if path == "step":
        s = _prepare_step(c, seed)
    elif path == "hess":
        s = _prepare_hess(c, seed)
    elif path == "update":
        s = _prepare_update(c, seed)
    elif path == "levels":
        s = dict(c=c, lv=[], src=[], rec=[], syn=[])
        for l, q in enumerate(_level_cases(c)):
            r, m = _inputs(q, seed + l)
            G = _geom(q, q["nt"])
            s["lv"].append(_context(ig.BatchContext, q, m, G, q["nt"], c["shots"], 1, c["ntr"]))
            shots = [_shot(q, r, q["nt"]) for _ in range(c["shots"])]
            s["src"].append([x[0] for x in shots])
            s["rec"].append([x[1] for x in shots])
            s["syn"].append(torch.zeros((c["shots"], 3, c["ntr"], q["nt"] + 1), device=DEV))
    else:
        r, m = _inputs(c, seed)
        nt = c["nt"]
        G = _geom(c, nt)
        n = c.get("shots", 1)
        shots = [_shot(c, r, nt) for _ in range(n)]
        s = dict(c=c, G=G, src=[x[0] for x in shots], rec=[x[1] for x in shots])
        s["obs"] = [torch.from_numpy(x[2]).to(DEV) for x in shots]
        if path == "batch":
            s["ctx"] = _context(ig.BatchContext, c, m, G, nt, n, c["nf"], c["ntr"])
        else:
            s["ctx"] = _context(ig.ShotContext, c, m, G, nt, c.get("nf", 1), c["ntr"])
        s["syn"] = torch.zeros(((n,) if path == "batch" else ()) + (3, c["ntr"], nt + 1), device=DEV)
        s["grad"] = [torch.zeros(G.dshape, device=DEV) for _ in range(3)] if c.get("adjoint", True) else None
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
NT_STEP = 40  # the time step of the "step" cases: near the wavelet's peak


def _run_step(s):
    c, G, f, m = s["c"], s["G"], s["f"], s["m"]
    ig.update_v(G, ig.REGION_INTERIOR, f, m, s["prof"], s["ps"])
    ig.update_v(G, ig.REGION_CPML, f, m, s["prof"], s["ps"])
    for region in (ig.REGION_INTERIOR, ig.REGION_CPML):
        if s["L"]:
            ig.update_s_visco(G, region, f, m, s["visco"], s["prof"], s["pv"])
        else:
            ig.update_s(G, region, f, m, s["prof"], s["pv"])
    ig.psource(G, f, s["src"], s["sig"], 1, NT_STEP)
    ig.discfourier(G, f, s["F"], s["C"], s["finv"], NT_STEP, 1, 0, ig.DFT_KAHAN if c["kahan"] else ig.DFT_COMPAT)
    if c["fs"]:
        ig.surface(G, f, m)
    ig.seismo(G, f, s["rec"], c["ntr"], NT_STEP, 200, s["sec"])
    return dict(f=f, ps=s["ps"], pv=s["pv"], F=s["F"], sec=s["sec"], r=s["r"] if s["L"] else [])


def _run_update(s):
    c, G, n = s["c"], s["G"], s["n"]
    g = s["work"]
    for a, b in zip(g, s["grad"]):
        ig.copy(a, b, n)
    ig.precon_grad(G, g, c["damp"], s["src"], s["rec"])
    for a, b in zip(s["test"], s["m"]):  # the line search's test model
        ig.copy(a, b, n)
    w = (1.0, 1.0, 0.5)
    if c["method"] == "lbfgs":
        h0 = s["lb"].update(g[0], g[1], 5)
        mx = ig.modelupdate(G, g, *s["test"], 0.02, w, 4000.0, 2300.0, 2000.0, bfgsmod=s["slot"], numpar=2)
        return dict(dir=g, model=s["test"], h0=np.float64(h0), maxima=mx)
    beta, _ = ig.conjugate(G, g, s["prior"], 0)
    mx = ig.modelupdate(G, g, *s["test"], 0.02, w, 4000.0, 2300.0, 2000.0)
    return dict(dir=g, model=s["test"], prior=s["prior"], beta=beta, maxima=mx)


def run(s):
    c = s["c"]
    path = c["path"]
    if path == "step":
        return _run_step(s)
    if path == "update":
        return _run_update(s)
    if path == "hess":
        for a in s["out"]:
            a.zero_()
        ig.gradient_F(s["G"], s["F"], s["B"], s["m"], s["finv"], s["out"][:3])
        ig.hess_F(s["G"], s["F"], s["B"], 1, s["m"], s["finv"], s["out"][3:])
        return dict(grad=s["out"][:3], hess=s["out"][3:])
    if path == "levels":
        ig.levels_run(s["lv"], s["src"], s["rec"], s["syn"], use_graph=True)
        return dict(syn=s["syn"])
    if path == "batch":
        if not c["adjoint"]:
            s["ctx"].run(s["src"], s["rec"], d_syn=s["syn"], want_adjoint=False, use_graph=c["graph"])
            return dict(syn=s["syn"])
        for a in s["grad"]:
            a.zero_()
        ig.sync()  # the batch runs on a stream of its own
        l2 = s["ctx"].run(s["src"], s["rec"], d_syn=s["syn"], grads=s["grad"], d_obs=s["obs"], use_graph=c["graph"])
        return dict(syn=s["syn"], grad=s["grad"], l2=np.array(l2))
    for a in s["grad"]:
        a.zero_()
    call = {"shot": s["ctx"].run_shot, "td": s["ctx"].run_shot_td, "adj": s["ctx"].run_shot_adj}[path]
    l2 = call(s["src"][0], s["rec"][0], s["syn"], s["grad"], d_obs=s["obs"][0])
    return dict(syn=s["syn"], grad=s["grad"], l2=np.float64(l2))


# ---------------------------------------------------------------------------
# what a pass cannot do without
def _cells(c):
    return float(c["nx"]) * c["ny"] * c["nz"]


def _step_work(c, shots=1):
    """one time step of `shots` shots: every wavefield (and memory variable)
    read and written once per update that changes it, the other operands
    read once, the model once for all shots; CPML memory of both updates"""
    n, L = _cells(c), c.get("L", 0)
    f2 = 2.0 * c["fw"]
    psi = f2 * (c["ny"] * c["nz"] + c["nx"] * c["nz"] + c["nx"] * c["ny"])
    b = shots * (n * (48.0 + 60.0 + 48.0 * L) + 2 * psi * 24.0) + n * (32.0 + (20.0 if L else 0.0))
    return b, shots * n * (75.0 + 85.0 + (40.0 * L + 40.0 if L else 0.0))


def _ntast(c, nt):
    return max(1, int(1.0 / (_finv(c, nt)[-1] * TAST * _dt(c))))


def work(case):
    c = dict(case)
    path = c["path"]
    if path == "levels":
        b = f = 0.0
        for q in _level_cases(c):
            x = _step_work(q, c["shots"])
            b, f = b + q["nt"] * x[0], f + q["nt"] * x[1]
        return {"bytes": b, "flops": f}
    n = _cells(c)
    if path == "hess":  # 12 DFT fields per frequency, the adjoint ones of two sets; model, two results
        return {"bytes": n * (4.0 * c["nf"] * 18 + 12.0 + 24.0), "flops": n * c["nf"] * 2 * 300.0}
    if path == "update":
        # gradients in, model in, direction and test model out; history of 4 pairs read and one gradient
        # and one step kept (L-BFGS), priors read and written (CG)
        hist = (8 * 2 + 4) * 4.0 if c["method"] == "lbfgs" else 12 * 4.0
        return {"bytes": n * (12.0 + 12.0 + 12.0 + 12.0 + hist), "flops": n * 120.0}
    x = _step_work(c, c.get("shots", 1))
    if path == "step":
        k = 2 if c["kahan"] else 1
        return {"bytes": x[0] + n * (12.0 + 48.0 * c["nf"] * k), "flops": x[1] + n * 12.0 * c["nf"]}
    nt, shots = c["nt"], c.get("shots", 1)
    if path == "batch" and not c["adjoint"]:
        return {"bytes": nt * x[0], "flops": nt * x[1]}
    if path in ("shot", "batch"):
        # the sampled velocities read once more, the DFT fields written once and read by the gradient
        samples = nt // _ntast(c, nt)
        return {"bytes": 2 * nt * x[0] + shots * n * (24.0 * samples + 96.0 * c["nf"]) + n * 24.0,
                "flops": 2 * nt * x[1] + shots * n * c["nf"] * (24.0 * samples + 300.0)}
    if path == "td":  # forward, recomputed forward, adjoint; both velocities read once more per sample
        return {"bytes": 3 * nt * x[0] + nt * n * 24.0, "flops": 3 * nt * x[1] + nt * n * 150.0}
    # forward, recomputed forward, the transposed step: the adjoint state as a step's, v and stress read again
    return {"bytes": 3 * nt * x[0] + nt * n * 36.0, "flops": 3 * nt * x[1] + nt * n * 200.0}


# ---------------------------------------------------------------------------
# the same in 64 bits: the scheme from its equations, in torch
class _Scheme:
    """The 4th-order staggered velocity-stress scheme with CPML on the grid
    of case c, in double.  Arrays are (y, x, z) with 3 cells before and 2
    after the grid; axes: 0 = y, 1 = x, 2 = z."""

    B1, B2 = 1.1382, -0.046414

    def __init__(self, c, m, nt):
        self.c, self.nt = c, nt
        self.n = (c["ny"], c["nx"], c["nz"])
        self.h, self.dt = c["dh"], float(np.float32(_dt(c)))
        self.fs = c.get("fs", 0)
        self.cpml(VPPML, _fpml(c, nt))
        self.model(*[m[n].to(torch.float64) for n in ("rho", "pi", "u")])
        self.L = c.get("L", 0)
        if self.L:
            t = self.wrap(m["taus"].to(torch.float64))
            self.taup, self.taus = self.at(m["taup"].to(torch.float64)), self.at(t)
            self.tau = {p: 0.25 * (self.at(t) + self.at(t, a) + self.at(t, b) + self.at(t, a, b))
                        for p, (a, b) in {"xy": (1, 0), "yz": (0, 2), "xz": (1, 2)}.items()}
            self.eta = m["eta"]

    # --- the model
    def at(self, f, *axes, by=1):
        """f at the grid's cells, moved by `by` cells along `axes`"""
        s = [slice(3 + (by if a in axes else 0), 3 + (by if a in axes else 0) + self.n[a]) for a in range(3)]
        return f[tuple(s)]

    def wrap(self, f):
        """periodic values one cell around the grid, as one rank's halo exchange leaves them"""
        i = torch.nn.functional.pad(self.at(f)[None, None], (1, 1, 1, 1, 1, 1), mode="circular")[0, 0]
        return torch.nn.functional.pad(i, (2, 1, 2, 1, 2, 1))

    def model(self, rho, pi, u):
        r, v = self.wrap(rho), self.wrap(u)
        self.rho, self.pi, self.u = self.at(rho), self.at(pi), self.at(u)
        self.rb = [0.5 * (self.at(r) + self.at(r, a)) for a in range(3)]  # between cells along y, x, z
        iv = 1.0 / torch.where(v == 0, torch.ones_like(v), v)
        self.mu = {p: 4.0 / (self.at(iv) + self.at(iv, a) + self.at(iv, b) + self.at(iv, a, b))
                   for p, (a, b) in {"xy": (1, 0), "yz": (0, 2), "xz": (1, 2)}.items()}

    # --- absorbing layers: K, a, b along each axis at cells and half cells
    def cpml(self, vp, f):
        fw, h, dt = self.c["fw"], self.h, self.dt
        d0 = -4.0 * vp * math.log(0.0008) / (2.0 * fw * h)
        side = {}
        for half in (0, 1):
            p = (fw - np.arange(1, fw + 2) + (0.5 if half else 1.0)) / fw
            d, K = d0 * (0.25 * p + 0.75 * p ** 3), 1.0 + p ** 3
            al = math.pi * f * (1.0 - p)
            b = np.exp(-(d / K + al) * dt)
            on = np.trunc(d) >= 1  # the coefficient a is left 0 where the whole part of d is
            a = np.where(on, d * (b - 1.0) / (K * (d + K * al)), 0.0)
            side[half] = (K, a, b, on)
        self.k = {}
        for half in (0, 1):
            K, a, b, _ = side[half]
            # the far side: half cells mirror the near side, cells lie one further out and start
            # with the layer's edge; a of both follows the cell profile's test
            on = side[0][3]
            if half:
                hi = K[fw - 1::-1], np.where(on[fw - 1::-1], a[fw - 1::-1], 0.0), b[fw - 1::-1]
            else:
                hi = K[fw:0:-1], a[fw:0:-1], b[fw:0:-1]
            for ax in range(3):
                v = [np.ones(self.n[ax]), np.zeros(self.n[ax]), np.zeros(self.n[ax])]
                for q, lo in enumerate((K, a, b)):
                    if not (ax == 0 and self.fs):
                        v[q][:fw] = lo[:fw]
                    v[q][-fw:] = hi[q]
                shape = [1, 1, 1]
                shape[ax] = self.n[ax]
                self.k[ax, half] = [torch.from_numpy(x).to(DEV).reshape(shape) for x in v]

    def damp(self, psi, d, ax, half):
        K, a, b = self.k[ax, half]
        p = b * psi + a * d
        return p, d / K + p

    # --- differences
    def fwd(self, f, ax):
        return self.B1 * (self.at(f, ax) - self.at(f)) + self.B2 * (self.at(f, ax, by=2) - self.at(f, ax, by=-1))

    def bwd(self, f, ax):
        return self.B1 * (self.at(f) - self.at(f, ax, by=-1)) + self.B2 * (self.at(f, ax) - self.at(f, ax, by=-2))

    def full(self, f):
        return torch.nn.functional.pad(f, (3, 2, 3, 2, 3, 2))

    def zero(self):
        """wavefields vx vy vz sxx syy szz sxy syz sxz, both CPML memories, memory variables"""
        z = [torch.zeros(self.n, dtype=torch.float64, device=DEV)]
        return [self.full(z[0])] * 9, z * 9, z * 9, [z * 6] * self.L

    # fields of a derivative: (field, forward difference, axis, CPML memory); half-cell profile = forward
    VD = ((3, 1, 1, 0), (6, 0, 0, 3), (8, 0, 2, 6), (4, 1, 0, 4), (6, 0, 1, 1), (7, 0, 2, 7), (5, 1, 2, 8),
          (8, 0, 1, 2), (7, 0, 0, 5))
    SD = ((0, 0, 1, 0), (0, 1, 0, 3), (0, 1, 2, 6), (1, 1, 1, 1), (1, 0, 0, 4), (1, 1, 2, 7), (2, 1, 1, 2),
          (2, 1, 0, 5), (2, 0, 2, 8))

    def velocity(self, f, ps, add=()):
        d, ps = [], list(ps)
        for n, fw, ax, q in self.VD:
            x = (self.fwd if fw else self.bwd)(f[n], ax) * (self.dt / self.h)
            ps[q], x = self.damp(ps[q], x, ax, fw)
            d.append(x)
        v = [self.at(f[0]) + (d[0] + d[1] + d[2]) / self.rb[1], self.at(f[1]) + (d[3] + d[4] + d[5]) / self.rb[0],
             self.at(f[2]) + (d[6] + d[7] + d[8]) / self.rb[2]]
        for n, idx, val in add:
            v[n] = v[n].index_put(idx, val, accumulate=True)
        return [self.full(x) for x in v] + list(f[3:]), ps

    def stress(self, f, pv, r, press=0.0, at=None):
        d, pv = [], list(pv)
        for n, fw, ax, q in self.SD:
            x = (self.fwd if fw else self.bwd)(f[n], ax) / self.h
            pv[q], x = self.damp(pv[q], x, ax, fw)
            d.append(x)
        xx, xy, xz, yx, yy, yz, zx, zy, zz = d
        dt, L = self.dt, self.L
        e = {"xy": xy + yx, "yz": yz + zy, "xz": xz + zx}
        tr = xx + yy + zz
        two = {"xx": yy + zz, "yy": xx + zz, "zz": xx + yy}
        gg, ff = self.pi, 2.0 * self.u
        if L:
            gg, ff = gg * (1.0 + L * self.taup), ff * (1.0 + L * self.taus)
        s = [self.at(f[3]) + dt * (gg * tr - ff * two["xx"]), self.at(f[4]) + dt * (gg * tr - ff * two["yy"]),
             self.at(f[5]) + dt * (gg * tr - ff * two["zz"])]
        for n, p in zip((6, 7, 8), ("xy", "yz", "xz")):
            s.append(self.at(f[n]) + self.mu[p] * dt * (1.0 + L * self.tau[p] if L else 1.0) * e[p])
        if L:
            new = []
            for l in range(L):
                eta = self.eta[l]
                b, cc = 1.0 / (1.0 + 0.5 * eta), 1.0 - 0.5 * eta
                ed = self.pi * eta * self.taup * tr
                dd = 2.0 * self.u * eta * self.taus
                q = [b * (r[l][n] * cc - ed + dd * two[p]) for n, p in enumerate(("xx", "yy", "zz"))]
                q += [b * (r[l][3 + n] * cc - self.mu[p] * eta * self.tau[p] * e[p])
                      for n, p in enumerate(("xy", "yz", "xz"))]
                for n in range(6):
                    s[n] = s[n] + 0.5 * dt * (r[l][n] + q[n])
                new.append(q)
            r = new
        if at is not None:
            for n in range(3):
                s[n] = s[n].index_put(at, torch.full((1,), press, dtype=torch.float64, device=DEV), accumulate=True)
        return list(f[:3]) + [self.full(x) for x in s], pv, r

    def surface(self, f):
        """a free surface at the first row: odd stresses above it, no vertical stress on it"""
        f = list(f)
        row = 3
        for n, off in ((4, 0), (6, 1), (7, 1)):
            f[n] = f[n].clone()
            if n == 4:
                f[n][row] = 0.0
            for m in (1, 2):
                f[n][row - m, 3:-2, 3:-2] = -f[n][row + m - off, 3:-2, 3:-2]
        v = [self.bwd(f[n], ax)[0] / self.h for n, ax in ((0, 1), (1, 0), (2, 2))]
        g, q = self.pi[0], self.pi[0] - 2.0 * self.u[0]
        hh = -(self.dt * q * q * (v[0] + v[2]) / g) - self.dt * q * v[1]
        for n in (3, 5):
            f[n] = f[n].clone()
            f[n][row, 3:-2, 3:-2] += hh
        return f

    # --- sources, receivers, records
    def wavelet(self, src):
        t = np.arange(self.nt + 2) * self.dt
        tau = math.pi * (t - 1.5 / src[4] - src[3]) * src[4]
        s = (1.0 - 2.0 * tau * tau) * np.exp(-tau * tau) * src[5]
        s[0] = s[self.nt + 1] = 0.0
        return s

    def spot(self, p):
        """index of grid positions [n][3] = x, y, z"""
        q = torch.as_tensor(np.atleast_2d(np.asarray(p, np.int64)) - 1).to(DEV)
        return q[:, 1], q[:, 0], q[:, 2]

    def pressure(self, sig, nt):
        hi = sig[nt + 1] if nt < self.nt else 0.0
        lo = sig[nt - 1] if nt > 1 else 0.0
        return (hi - lo) / (2.0 * self.h ** 3)

    def step(self, st, nt, src=None, sig=None, adj=None, rec=None):
        """one step: the source (forward) or the residuals, injected twice (adjoint)"""
        f, ps, pv, r = st
        add, at, press = [], None, 0.0
        if src is not None and src[6] > 1:
            n, k = {2: (0, 1), 3: (2, 0), 4: (1, 2)}[src[6]]  # component and its density average
            idx = self.spot(src[:3])
            add = [(n, idx, self.dt * sig[nt] / self.h ** 3 * self.rb[k][idx])]
        elif src is not None:
            at, press = self.spot(src[:3]), float(self.pressure(sig, nt))
        if adj is not None:
            add = [(n, rec, 2.0 * adj[n, :, nt]) for n in range(3)]
        f, ps = self.velocity(f, ps, add)
        f, pv, r = self.stress(f, pv, r, press, at)
        if self.fs:
            f = self.surface(f)
        return f, ps, pv, r

    def forward(self, src, rec, each=None):
        sig, idx, st = self.wavelet(src), self.spot(rec), self.zero()
        syn = torch.zeros((3, len(rec), self.nt + 1), dtype=torch.float64, device=DEV)
        for nt in range(1, self.nt + 1):
            st = self.step(st, nt, src, sig)
            for n in range(3):
                syn[n, :, nt] = self.at(st[0][n])[idx]
            if each:
                each(nt, st[0])
        return syn

    def residual(self, syn, obs):
        """time-reversed running sums of the residual, and the sum of their squares"""
        d = self.dt * torch.cumsum(syn[..., 1:] - obs.to(torch.float64)[..., 1:], -1)
        adj = torch.zeros_like(syn)
        adj[..., 1:] = d.flip(-1)
        return adj, float((d * d).sum())

    def adjoint(self, adj, rec, each, last=None):
        st, idx = self.zero(), self.spot(rec)
        for nt in range(1, (last or self.nt) + 1):
            st = self.step(st, nt, adj=adj, rec=idx)
            each(nt, st[0])

    def strain(self, f):
        """the nine derivatives of three fields (padded)"""
        return [(self.fwd if fw else self.bwd)(f[n], ax) / self.h for n, fw, ax, _ in self.SD]


def _products(a, b):
    """(tr a tr b, the shear-modulus product) of two strain sets"""
    lam = (a[0] + a[4] + a[8]) * (b[0] + b[4] + b[8])
    mu = 2 * (a[0] * b[0] + a[4] * b[4] + a[8] * b[8]) + (a[1] + a[3]) * (b[1] + b[3])
    mu = mu + (a[2] + a[6]) * (b[2] + b[6]) + (a[5] + a[7]) * (b[5] + b[7])
    return lam, mu


def _to_vp_vs_rho(S, lam, mu, rho):
    """gradients of vp, vs, rho from those of lambda, mu and the density term"""
    sp, su = torch.sqrt(S.rho * S.pi), torch.sqrt(S.rho * S.u)
    return [2 * sp * lam, -4 * su * lam + 2 * su * mu, rho + S.u / S.rho * mu + (S.pi - 2 * S.u) / S.rho * lam]


def _freq_gradient(S, F, B, finv):
    """F, B: [nf][6] padded fields (re x y z, im x y z)"""
    out = [0.0, 0.0, 0.0]
    for l, f in enumerate(finv):
        w = 1.0 / (4.0 * math.pi ** 2 * f * f)
        lam = mu = rho = 0.0
        for o in (0, 3):
            a, b = S.strain(F[l][o:o + 3]), S.strain(B[l][o:o + 3])
            x, y = _products(a, b)
            lam, mu = lam - w * x, mu - w * y
            rho = rho + sum(S.at(F[l][o + n]) * S.at(B[l][o + n]) for n in range(3))
        out = [p + q for p, q in zip(out, _to_vp_vs_rho(S, lam, mu, rho))]
    return out


def _freq_hessian(S, F, B, finv):
    out = [0.0, 0.0, 0.0]
    for l, f in enumerate(finv):
        w = 1.0 / (2.0 * math.pi * f)
        a, ai = S.strain(F[l][:3]), S.strain(F[l][3:])
        b, bi = S.strain(B[l][:3]), S.strain(B[l][3:])
        aibr, arbi, aibi, arbr = _products(ai, b), _products(a, bi), _products(ai, bi), _products(a, b)
        relam, remu = w * (aibr[0] + arbi[0]), w * (aibr[1] + arbi[1])
        imlam, immu = w * (aibi[0] - arbr[0]), w * (aibi[1] - arbr[1])
        dot = lambda p, q: sum(S.at(F[l][p + n]) * S.at(B[l][q + n]) for n in range(3))  # noqa: E731
        rer, imr = dot(0, 0) - dot(3, 3), dot(0, 3) + dot(3, 0)
        rer = rer + relam * (S.pi - 2 * S.u) / S.rho + remu * S.u / S.rho
        imr = imr + imlam * (S.pi - 2 * S.u) / S.rho + immu * S.u / S.rho
        rv, iv = remu - 2 * relam, immu - 2 * imlam
        out = [out[0] + 4 * (relam ** 2 + imlam ** 2) * S.rho * S.pi, out[1] + 4 * (rv ** 2 + iv ** 2) * S.rho * S.u,
               out[2] + rer ** 2 + imr ** 2]
    return out


def _pitched(c, a):
    """values of the grid's cells in the device layout"""
    pitch = (c["nz"] + ig.KOFF + 3 + 31) // 32 * 32
    return torch.nn.functional.pad(a, (ig.KOFF + 1, pitch - ig.KOFF - 1 - c["nz"], 3, 2, 3, 2))


def _padded(c, a):
    """a field of the device layout as the scheme's padded double array"""
    return a[..., ig.KOFF - 2:ig.KOFF - 2 + c["nz"] + 5].to(torch.float64)


class _Dft:
    def __init__(self, S, finv):
        self.S, self.finv, self.ntast = S, finv, _ntast(S.c, S.nt)
        self.F = [[torch.zeros(S.n, dtype=torch.float64, device=DEV) for _ in range(6)] for _ in finv]

    def add(self, nt, f, back):
        if nt % self.ntast:
            return
        S = self.S
        t = (S.nt - 1 - nt) * S.dt if back else nt * S.dt
        for F, fr in zip(self.F, self.finv):
            for n in range(3):
                v = S.at(f[n])
                F[n] += v * (math.cos(2 * math.pi * fr * t) * S.dt * self.ntast)
                F[3 + n] += v * (math.sin(2 * math.pi * fr * t) * S.dt * self.ntast)

    def full(self):
        return [[self.S.full(x) for x in F] for F in self.F]


def _exact_shot(c, m, src, rec, obs, nt):
    S = _Scheme(c, m, nt)
    fwd, bwd = _Dft(S, _finv(c, nt)), _Dft(S, _finv(c, nt))
    syn = S.forward(src, rec, lambda n, f: fwd.add(n, f, 0))
    adj, l2 = S.residual(syn, torch.from_numpy(obs).to(DEV))
    S.adjoint(adj, rec, lambda n, f: bwd.add(n, f, 1))
    return syn, _freq_gradient(S, fwd.full(), bwd.full(), fwd.finv), l2


def _exact_td(c, m, src, rec, obs, nt):
    """the full-band gradient: displacements integrated from the record's end"""
    S = _Scheme(c, m, nt)
    hist = []
    syn = S.forward(src, rec, lambda n, f: hist.append(f[:3]))
    adj, l2 = S.residual(syn, torch.from_numpy(obs).to(DEV))
    uf = [S.dt * (hist[nt - 1][q] + hist[nt - 2][q]) for q in range(3)]
    ub = [torch.zeros_like(x) for x in uf]
    acc = [0.0, 0.0, 0.0]

    def each(step, f):
        vf = hist[nt - 2 - step]
        for q in range(3):
            uf[q] = uf[q] + S.dt * vf[q]
            ub[q] = ub[q] + S.dt * f[q]
        lam, mu = _products(S.strain(uf), S.strain(ub))
        acc[0] = acc[0] - S.dt * lam
        acc[1] = acc[1] - S.dt * mu
        acc[2] = acc[2] + S.dt * sum(S.at(vf[q]) * S.at(f[q]) for q in range(3))

    S.adjoint(adj, rec, each, nt - 2)
    return syn, _to_vp_vs_rho(S, *acc), l2


def _exact_adj(c, m, src, rec, obs, nt):
    """the misfit's derivative by reverse differentiation of the scheme"""
    from torch.utils.checkpoint import checkpoint
    S = _Scheme(c, m, nt)
    rho = m["rho"].to(torch.float64)
    vp, vs = torch.sqrt(m["pi"].to(torch.float64) / rho), torch.sqrt(m["u"].to(torch.float64) / rho)
    x = [a.detach().requires_grad_(True) for a in (vp, vs, rho)]
    obs = torch.from_numpy(obs).to(DEV, torch.float64)
    sig, idx, st = S.wavelet(src), S.spot(rec), S.zero()

    def step(nt, f, ps, pv, vp, vs, rho):
        S.model(rho, rho * vp * vp, rho * vs * vs)
        f, ps, pv, _ = S.step((f, ps, pv, []), nt, src, sig)
        return f, ps, pv, torch.stack([S.at(f[n])[idx] for n in range(3)])

    f, ps, pv, _ = st
    syn, J = torch.zeros((3, len(rec), nt + 1), dtype=torch.float64, device=DEV), 0.0
    for n in range(1, nt + 1):
        f, ps, pv, s = checkpoint(step, n, f, ps, pv, *x, use_reentrant=False)
        syn[..., n] = s.detach()
        J = J + 0.5 * ((s - obs[..., n]) ** 2).sum()
    g = torch.autograd.grad(J, x)
    return syn, [S.at(a).detach() for a in g], float(J.detach())


def _exact_step(c, seed):
    r, m = _inputs(c, seed)
    S = _Scheme(c, m, 200)
    fields = [_field(r, c, n).to(torch.float64) for n in range(9)]
    src, rec, _ = _shot(c, r, 200)
    _, ps, pv, mem = S.zero()
    f, ps = S.velocity(fields, ps)
    f, pv, mem = S.stress(f, pv, mem, float(S.pressure(S.wavelet(src), NT_STEP)), S.spot(src[:3]))
    F = []
    for trig in (math.cos, math.sin):
        for n in range(3):
            F.append(torch.stack([_pitched(c, S.at(f[n]) * (trig(2 * math.pi * q * NT_STEP * S.dt) * S.dt))
                                  for q in _finv(c, 200)]))
    if c["fs"]:
        f = S.surface(f)
    sec = torch.zeros((3, c["ntr"], 201), dtype=torch.float64, device=DEV)
    for n in range(3):
        sec[n, :, NT_STEP] = S.at(f[n])[S.spot(rec)]

    def slabs(p, n):
        ax, fw = (1, 0, 2)[n // 3], c["fw"]
        return torch.cat([p.narrow(ax, 0, fw), p.narrow(ax, S.n[ax] - fw, fw)], ax)

    pitch = (c["nz"] + ig.KOFF + 3 + 31) // 32 * 32
    dev = lambda a: torch.nn.functional.pad(a, (ig.KOFF - 2, pitch - ig.KOFF + 2 - c["nz"] - 5))  # noqa: E731
    return dict(f=[dev(a) for a in f], ps=[slabs(p, n) for n, p in enumerate(ps)],
                pv=[slabs(p, n) for n, p in enumerate(pv)], F=F, sec=sec,
                r=[torch.stack([_pitched(c, mem[l][n]) for l in range(c["L"])]) for n in range(6)] if c["L"] else [])


def _taper(c, src, rec):
    """the product of the source, receiver and edge tapers on the grid's cells"""
    j, i, k = [torch.arange(1, n + 1, device=DEV, dtype=torch.float64) for n in (c["ny"], c["nx"], c["nz"])]
    on = c["damp"] in (1, 2)
    if not on:
        j, i, k = j * 0, i * 0, k * 0
    t = torch.ones((c["ny"], c["nx"], c["nz"]), dtype=torch.float64, device=DEV)
    if c["damp"] == 2:
        for x, y, z in src:
            r = torch.sqrt((j - y)[:, None, None] ** 2 + (i - x)[:, None] ** 2 + (k - z) ** 2)
            t = t / (1.0 + 1000.0 * torch.exp(-0.7 * r))
    if on:
        for x, y, z in rec:  # 1 within 1e-16 beyond 8 cells
            b = [slice(max(0, p - 10), p + 9) for p in (int(y), int(x), int(z))]
            r2 = (j[b[0]] - y)[:, None, None] ** 2 + (i[b[1]] - x)[:, None] ** 2 + (k[b[2]] - z) ** 2
            t[tuple(b)] /= 1.0 + 1000.0 * torch.exp(-0.7 * r2)
    for a, n, s in ((j, c["ny"], (-1, 1, 1)), (i, c["nx"], (1, -1, 1)), (k, c["nz"], (1, 1, -1))):
        e = 1.0 / (1.0 + 2000.0 * torch.exp(-0.6 * a)) / (1.0 + 2000.0 * torch.exp(-0.6 * (n - a)))
        t = t * e.reshape(s)
    return t


def _exact_update(c, seed):
    m, g, s, src, rec = _update_inputs(c, seed)
    T = _taper(c, src, rec)
    g = [a.to(torch.float64) * T for a in g]
    d = g[4].clone()
    out = {}
    if c["method"] == "lbfgs":
        y = [g[n][:2] - g[n + 1][:2] for n in range(4)]
        s = [a.to(torch.float64) for a in s]
        ys = [float((a * b).sum()) for a, b in zip(y, s)]
        h0 = ys[3] / float((y[3] * y[3]).sum())
        q, al = g[4][:2].clone(), [0.0] * 4
        for n in (3, 2, 1, 0):
            al[n] = float((s[n] * q).sum()) / ys[n]
            q -= al[n] * y[n]
        q *= h0
        for n in range(4):
            q += s[n] * (al[n] - float((y[n] * q).sum()) / ys[n])
        d[:2] = q
        out["h0"] = np.float64(h0)
    else:
        p = g[3]
        beta = [float((g[4][n] * (g[4][n] - p[n])).sum() / (p[n] * p[n]).sum()) for n in range(3)]
        beta[0] = min(max(beta[0], 0.0), 0.5)
        d = torch.stack([p[n] * beta[n] + g[4][n] for n in range(3)])
        out["prior"] = [_pitched(c, a) for a in g[4]] + [_pitched(c, a) for a in d]
        out["beta"] = np.array(beta)
    rho, pi, u = [m[n].to(torch.float64)[3:-2, 3:-2, 3:-2] for n in ("rho", "pi", "u")]
    vp, vs = torch.sqrt(pi / rho), torch.sqrt(u / rho)
    if c["method"] == "cg":
        d = torch.stack([d[n] / d[n].abs().max() for n in range(3)])
    vn, sn, rn = vp + 0.02 * d[0] * 4000.0, vs + 0.02 * d[1] * 2300.0, rho + 0.01 * d[2] * 2000.0
    full = [m[n].to(torch.float64).clone() for n in ("rho", "pi", "u")]
    for a, b in zip(full, (rn, rn * vn * vn, rn * sn * sn)):
        a[3:-2, 3:-2, 3:-2] = b
    pitch = (c["nz"] + ig.KOFF + 3 + 31) // 32 * 32
    out["model"] = [torch.nn.functional.pad(a, (ig.KOFF - 2, pitch - ig.KOFF + 2 - c["nz"] - 5)) for a in full]
    out["dir"] = [_pitched(c, a) for a in d]
    out["maxima"] = np.array([float(vp.max()), float(vs.max()), float(rho.max())])
    return out


#: cell-steps of a whole propagation that the scheme in torch does in about 20 seconds
MOST = 4.5e9


def exact(case, seed):
    c = dict(case)
    path = c["path"]
    if path == "step":
        return _exact_step(c, seed)
    if path == "update":
        return _exact_update(c, seed)
    if path == "hess":
        s = _prepare_hess(c, seed)
        S = _Scheme(c, _inputs(c, seed)[1], 100)
        nf = c["nf"]
        F = [[_padded(c, s["F"][n][l]) for n in range(6)] for l in range(nf)]
        B = [[_padded(c, s["B"][n][l]) for n in range(6)] for l in range(2 * nf)]
        return dict(grad=[_pitched(c, a) for a in _freq_gradient(S, F, B[:nf], s["finv"])],
                    hess=[_pitched(c, a) for a in _freq_hessian(S, F, B[nf:], s["finv"])])
    if path == "levels":
        syn = []
        for l, q in enumerate(_level_cases(c)):
            r, m = _inputs(q, seed + l)
            shots = [_shot(q, r, q["nt"]) for _ in range(c["shots"])]
            S = _Scheme(q, m, q["nt"])
            syn.append(torch.stack([S.forward(x[0], x[1]) for x in shots]))
        return dict(syn=syn)
    shots, nt = c.get("shots", 1), c["nt"]
    passes = 1 if not c.get("adjoint", True) else 2
    if _cells(c) * nt * passes * shots * (2.0 if c.get("L") else 1.0) > MOST:
        return None
    r, m = _inputs(c, seed)
    got = [_shot(c, r, nt) for _ in range(shots)]
    if passes == 1:
        S = _Scheme(c, m, nt)
        return dict(syn=torch.stack([S.forward(x[0], x[1]) for x in got]))
    call = {"shot": _exact_shot, "batch": _exact_shot, "td": _exact_td, "adj": _exact_adj}[path]
    res = [call(c, m, *x, nt) for x in got]
    grad = [_pitched(c, sum(x[1][n] for x in res)) for n in range(3)]
    if path == "batch":
        return dict(syn=torch.stack([x[0] for x in res]), grad=grad, l2=np.array([x[2] for x in res]))
    return dict(syn=res[0][0], grad=grad, l2=np.float64(res[0][2]))
