"""Performance cases of upcgen_amd: the calls that its users' programs spend
their time in, over the range of sizes they are made at.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges; `prepare(case, seed)` makes what a program holds
before the call (contexts, batches, networks, tables; configurations and data
vary with the seed), `run(state)` is one call sequence, `work(case)` its
algorithmic bytes and operations, `exact(case, seed)` the outputs in plain
64-bit torch where they have a value independent of the library.
"""
import math
import random

import numpy as np
import torch

import upcgen_amd as U
from upcgen_amd import surrogate as S

# Collision systems: Z, A, R [fm], a [fm], sqrt(s_NN) [GeV]
SYSTEMS = {
    "pb": (82, 208, 6.68, 0.447, 5020.0),
    "xe": (54, 129, U.wood_saxon_radius(129), 0.54, 5440.0),
    "au": (79, 197, U.wood_saxon_radius(197), 0.54, 200.0),
    "o": (8, 16, U.wood_saxon_radius(16), 0.54, 7000.0),
}


def listed():
    return [
        # A program asks for L at a few scattered (M, Y): the smallest call, all latency.
        dict(name="points_33_form", kind="points", system="pb", mode=2, flux_point=0, pol=0, n=33),
        # Scattered quadrature labels of one system, as the surrogate's data sets are made of.
        dict(name="points_4096_form", kind="points", system="xe", mode=4, flux_point=0, pol=0, n=4096),
        # The small plain grid: point-charge flux, no breakup factor.
        dict(name="grid_101x41_point", kind="grid", system="pb", mode=1, flux_point=1, pol=0, form="fp64",
             nm=101, ny=41, ymin=-6.0, ymax=6.0),
        # The package's default grid (point-charge flux at full size).
        dict(name="grid_1001x121_point", kind="grid", system="pb", mode=1, flux_point=1, pol=0, form="fp64",
             nm=1001, ny=121, ymin=-6.0, ymax=6.0),
        # A polarised light-ion grid on one-sided rapidities (no mirror bins), form-factor flux.
        dict(name="grid_251x41_form_pol", kind="grid", system="o", mode=3, flux_point=0, pol=1, form="fp64",
             nm=251, ny=41, ymin=-1.5, ymax=4.5),
        # The matrix form of the contraction on an odd grid.
        dict(name="grid_1501x81_mfma", kind="grid", system="xe", mode=4, flux_point=1, pol=0, form="mfma",
             nm=1501, ny=81, ymin=-6.0, ymax=6.0),
        # One configuration from init to the sampler tables (UpcGenerator::init -> computeNuclXsection).
        dict(name="step_1001x121_form", kind="step", system="pb", mode=2, nm=1001, ny=121, nz=100,
             ymin=-6.0, ymax=6.0, proc=13),
        # A serving batch of mixed systems and uneven grids, replayed from its graph.
        dict(name="batch_16", kind="batch", jobs=16, jobs_seed=2024, flux_point=0, pol=1),
        # The form-factor flux at points of a program's own choosing.
        dict(name="flux_50021", kind="flux", system="pb", n=50021),
        # Event generation: (Y, M, z) draws from the tables, then whole lepton pairs.
        dict(name="draws_16777259", kind="draws", nm=1001, ny=121, nz=100, pol=0, n=16777259, proc=15),
        dict(name="pairs_2000003", kind="pairs", nm=1001, ny=121, nz=100, pol=0, n=2000003, proc=13, gampt=1),
        # One forward and backward pass of the surrogate's two networks, and its inference.
        dict(name="net_8192", kind="net", rows=8192, infer=121121),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "grid", "grid", "grid", "step", "batch", "flux", "draws", "pairs", "net"])
    system = rng.choice(sorted(SYSTEMS))
    mode = rng.randint(1, 4)
    if kind == "points":
        return dict(kind=kind, system=system, mode=mode, flux_point=rng.choice([0, 0, 1]), pol=rng.choice([0, 0, 1]),
                    n=_logint(rng, 1, 20000))
    if kind in ("grid", "step"):
        nm, ny = _logint(rng, 21, 1001), _logint(rng, 11, 121)
        y = rng.choice([(-6.0, 6.0), (-6.0, 6.0), (-4.0, 4.0), (-1.5, 4.5)])
        if kind == "step":
            return dict(kind=kind, system=system, mode=mode, nm=nm, ny=ny, nz=rng.randint(20, 100), ymin=y[0],
                        ymax=y[1], proc=rng.choice([11, 13]))
        return dict(kind=kind, system=system, mode=mode, flux_point=rng.choice([0, 1]), pol=rng.choice([0, 0, 1]),
                    form=rng.choice(["fp64", "fp64", "mfma"]), nm=nm, ny=ny, ymin=y[0], ymax=y[1])
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 8), jobs_seed=rng.randint(1, 10 ** 6),
                    flux_point=rng.choice([0, 0, 1]), pol=rng.choice([0, 1]))
    if kind == "flux":
        return dict(kind=kind, system=system, n=_logint(rng, 1, 200000))
    if kind == "net":
        return dict(kind=kind, rows=64 * _logint(rng, 1, 256), infer=_logint(rng, 33, 121121))
    return dict(kind=kind, nm=_logint(rng, 21, 1001), ny=_logint(rng, 11, 121), nz=rng.randint(20, 100),
                pol=rng.choice([0, 1]), n=_logint(rng, 1000, 16777259 if kind == "draws" else 4000000),
                proc=rng.choice([13, 15]), **({"gampt": rng.choice([0, 1])} if kind == "pairs" else {}))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _config(case, seed, **kw):
    """The case's configuration with radius and mass range a little different for every seed."""
    r = random.Random(1000003 * seed + 17)
    Z, A, R, a, sqrts = SYSTEMS[case.get("system", "pb")]
    mmin = 3.56 if case.get("proc", 13) == 15 else 3.5
    v = dict(Z=Z, A=A, R=R * r.uniform(0.98, 1.02), a=a, sqrts=sqrts, flux_point=case.get("flux_point", 0),
             breakup_mode=case.get("mode", 1), use_polarized=case.get("pol", 0),
             mmin=mmin * r.uniform(1.0, 1.02), mmax=50.0 * r.uniform(0.98, 1.0), proc_id=case.get("proc", 13))
    for k in ("nm", "ny", "nz", "ymin", "ymax"):
        if k in case:
            v[k] = case[k]
    v.update(kw)
    return U.Config.make(**v)


def _gen(seed):
    return np.random.default_rng(7919 * seed + 5)


def _points(case, seed):
    rng = _gen(seed)
    M = np.exp(rng.uniform(math.log(1.0), math.log(100.0), case["n"]))
    return torch.from_numpy(M), torch.from_numpy(rng.uniform(-5.0, 5.0, case["n"]))


def _cdf(w):
    """Prefix sums over the last axis, normalised: [..., n + 1] from 0 to 1."""
    c = np.cumsum(w, axis=-1)
    c = c / c[..., -1:]
    return torch.from_numpy(np.concatenate([np.zeros(c.shape[:-1] + (1,)), c], axis=-1))


def _tables(case, seed, cfg):
    """Sampler tables of the shape a cross-section grid has: falling in M, bell-shaped in Y, peaked at |z| = 1."""
    rng = _gen(seed)
    nm, ny, nz = case["nm"], case["ny"], case["nz"]
    M = np.linspace(cfg.mmin, cfg.mmax, nm, endpoint=False)
    Y = np.linspace(cfg.ymin, cfg.ymax, ny, endpoint=False)
    z = np.linspace(cfg.zmin, cfg.zmax, nz, endpoint=False) + 1.0 / nz
    t = dict(sum_ym=_cdf((np.exp(-Y[:, None] ** 2 / 9.0) * M[None, :] ** -4.5
                          * rng.uniform(0.5, 1.5, (ny, nm))).reshape(-1)))
    zw = lambda p: _cdf((1.0 / (1.0 - np.minimum(z * z, 0.9999)))[None, :] ** p * rng.uniform(0.5, 1.5, (nm, nz)))
    if case["pol"]:
        t.update(sum_zs=zw(1.0), sum_zp=zw(0.5), ratio=torch.from_numpy(rng.uniform(0.2, 0.8, (ny, nm))))
    else:
        t.update(sum_z=zw(1.0))
    return t


NET_SHAPES = ((128, 32), (128,), (128, 128), (128,), (128, 128), (128,), (128,), (1,))


def _net(case, seed):
    """Weights of two networks, features, baseline logs and targets."""
    rng = _gen(seed)
    nets = []
    for _ in range(2):
        nets.append(np.concatenate([(rng.standard_normal(s) * (1.2 / math.sqrt(s[-1]) if len(s) == 2 else 0.1)).ravel()
                                    for s in NET_SHAPES]).astype(np.float32))
    n = max(case["rows"], case["infer"])
    X = np.zeros((n, 32), dtype=np.float32)
    X[:, :13] = rng.uniform(-1.5, 1.5, (n, 13))
    return nets, X, rng.uniform(-20.0, 5.0, n), rng.standard_normal(n).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "points":
        M, Y = _points(case, seed)
        return dict(kind=kind, ctx=U.Context(_config(case, seed)), M=M.cuda(), Y=Y.cuda())
    if kind == "grid":
        return dict(kind=kind, ctx=U.Context(_config(case, seed)),
                    form={"fp64": U.FORM_FP64, "mfma": U.FORM_MFMA}[case["form"]])
    if kind == "step":
        return dict(kind=kind, ctx=U.Context(_config(case, seed)))
    if kind == "batch":
        r = random.Random(1000003 * seed + 29)
        jobs = U.mixed_systems_jobs(seed=case["jobs_seed"], n=case["jobs"], polarized=case["pol"],
                                    flux_point=case["flux_point"])
        for c in jobs:
            c.R *= r.uniform(0.98, 1.02)
        return dict(kind=kind, batch=U.Batch(jobs))
    if kind == "flux":
        cfg = _config(case, seed)
        rng = _gen(seed)
        b = rng.uniform(0.05 * cfg.R, 2.5 * cfg.R, case["n"])
        k = np.exp(rng.uniform(math.log(0.01), math.log(300.0 * cfg.sqrts / 5020.0), case["n"]))
        return dict(kind=kind, ctx=U.Context(cfg), b=torch.from_numpy(b).cuda(), k=torch.from_numpy(k).cuda())
    if kind in ("draws", "pairs"):
        cfg = _config(case, seed)
        ctx = U.Context(cfg)
        st = dict(kind=kind, ctx=ctx, n=case["n"], seed=12345 + seed,
                  tables={k: t.cuda() for k, t in _tables(case, seed, cfg).items()})
        if kind == "pairs":
            st["opts"] = U.EventOpts(case["gampt"], 1, 1.0, 1, -2.5, 2.5)
            if case["gampt"]:
                ctx.photon_pt_tables(ctx.info.g1)
        return st
    nets, X, L0, T = _net(case, seed)
    s = S.Surrogate(1)
    for i in range(2):
        s.set_params(i, nets[i])
    s.norm = (0.1, 0.7)
    X = torch.from_numpy(X).cuda()
    return dict(kind=kind, sur=s, X=X[:case["infer"]].contiguous(), L0=torch.from_numpy(L0[:case["infer"]]).cuda(),
                Xb=X[:case["rows"]].contiguous(), T=torch.from_numpy(T[:case["rows"]]).cuda())


def run(st):
    kind = st["kind"]
    if kind == "points":
        return st["ctx"].lumi_points(st["M"], st["Y"])
    if kind == "grid":
        return st["ctx"].lumi_grid(st["form"])
    if kind == "step":
        ctx = st["ctx"]
        ctx.rebuild_tables()
        # bins whose flux integrals leave the form-factor table are NaN: no cross section there
        L = torch.nan_to_num(ctx.lumi_grid(), nan=0.0)
        zm = ctx.cs_zm()
        cs, _, tot = ctx.nuc_cs_ym(L)
        return dict(zm=zm, sum_z=ctx.pdf_init(zm), L=L, cs=cs, sum_ym=ctx.pdf_init(cs.reshape(1, -1)), tot=tot)
    if kind == "batch":
        return st["batch"].run(graph=True)
    if kind == "flux":
        return st["ctx"].flux_form(st["b"], st["k"])
    if kind == "draws":
        return st["ctx"].sample_events(**st["tables"], n=st["n"], seed=st["seed"])
    if kind == "pairs":
        return st["ctx"].generate_pairs(**st["tables"], n=st["n"], seed=st["seed"], opts=st["opts"])
    s = st["sur"]
    return s.log_lumi(st["X"], st["L0"]), s.grad(0, st["Xb"], st["T"]), s.grad(1, st["Xb"], st["T"])


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
FLOP_POINT = 173040           # node contraction of one unpolarised (M, Y) bin
FLOP_INTEGRAL = 290 * 132     # one form-factor flux integral: integrand evaluations x their operations
INTEGRALS_ROW = 69            # form-factor nodes of a flux row


def _lumi_flops(npts, rows, flux_point, pol):
    return npts * FLOP_POINT * (2 if pol else 1) + rows * (120 * 120 if flux_point else INTEGRALS_ROW * FLOP_INTEGRAL)


def work(case):
    kind = case["kind"]
    if kind == "points":
        n, pol = case["n"], case["pol"]
        return dict(bytes=8 * n * (3 + pol), flops=_lumi_flops(n, 2 * n, case["flux_point"], pol))
    if kind in ("grid", "step"):
        n, pol = case["nm"] * case["ny"], case.get("pol", 0)
        sym = case["ymin"] == -case["ymax"]
        rows = n + case["nm"] if sym else 2 * n
        w = dict(bytes=8 * n * (1 + pol), flops=_lumi_flops(n, rows, case.get("flux_point", 0), pol))
        if kind == "step":
            w["bytes"] += 8 * n * 2 + 16 * case["nm"] * case["nz"] + 32000000
            w["flops"] += 1000000 * 200 + 20096 * 600 * 60
        return w
    if kind == "batch":
        jobs = U.mixed_systems_jobs(seed=case["jobs_seed"], n=case["jobs"], polarized=case["pol"],
                                    flux_point=case["flux_point"])
        n = sum(c.nm * c.ny for c in jobs)
        rows = n + sum(c.nm for c in jobs)
        return dict(bytes=8 * n * (1 + case["pol"]), flops=_lumi_flops(n, rows, case["flux_point"], case["pol"]))
    if kind == "flux":  # b uniform in [0.05, 2.5] R: 80 % of the points lie inside 2R
        return dict(bytes=28 * case["n"], flops=int(0.8 * case["n"] * FLOP_INTEGRAL))
    if kind in ("draws", "pairs"):
        tab = 8 * case["nm"] * (case["ny"] * (1 + case["pol"]) + case["nz"] * (1 + case["pol"]))
        return dict(bytes=(24 if kind == "draws" else 76) * case["n"] + tab,
                    flops=(200 if kind == "draws" else 900) * case["n"])
    mac = 32 * 128 + 2 * 128 * 128 + 128
    return dict(bytes=case["infer"] * (128 + 24) + 2 * case["rows"] * 132 + 6 * 4 * 37377,
                flops=2 * 2 * mac * (case["infer"] + 3 * case["rows"]))


# ---------------------------------------------------------------------------
# Values in 64 bits, without the library
# ---------------------------------------------------------------------------
HC, MP = 0.1973269718, 0.9382720813
ALPHA = 1.0 / 137.035999074
GLX = (0.1488743389816312, 0.4333953941292472, 0.6794095682990244, 0.8650633666889845, 0.9739065285171717)
GLW = (0.2955242247147529, 0.2692667193099963, 0.2190863625159820, 0.1494513491505806, 0.0666713443086881)


def _simpson_w(n, h):
    w = np.zeros(n)
    w[0] = w[-1] = 1.0
    w[1:n - 1:2] = 4.0
    w[2:n - 1:2] = 2.0
    return w * h / 3.0


class _Spline:
    """Natural cubic spline on uniform knots from 0."""

    def __init__(self, y, h, dev):
        n = len(y)
        A = np.zeros((n, n))
        rhs = np.zeros(n)
        A[0, 0] = A[-1, -1] = 1.0
        for i in range(1, n - 1):
            A[i, i - 1:i + 2] = (1.0, 4.0, 1.0)
            rhs[i] = 3.0 * (y[i + 1] - 2.0 * y[i] + y[i - 1]) / (h * h)
        c = np.linalg.solve(A, rhs)
        b = (y[1:] - y[:-1]) / h - h * (c[1:] + 2.0 * c[:-1]) / 3.0
        d = (c[1:] - c[:-1]) / (3.0 * h)
        self.h, self.n = h, n
        self.t = [torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in (y[:-1], b, c[:-1], d)]

    def __call__(self, x):
        i = (x / self.h).long().clamp_(0, self.n - 2)
        u = x - i.double() * self.h
        y, b, c, d = (v[i] for v in self.t)
        return y + u * (b + u * (c + u * d))


def _overlap(cfg, dev):
    """G_AA(b) on [0, 20] fm: the optical Glauber factor on its 200 knots."""
    n, h = 200, 20.0 / 199
    w = _simpson_w(n, h)
    r = np.arange(n) * h
    ws = lambda x: 1.0 / (1.0 + np.exp((x - cfg.R) / cfg.a))
    rho0 = cfg.A / float(w @ (r * r * ws(r))) / 4.0 / math.pi
    ta = _Spline(2.0 * rho0 * (ws(np.sqrt(r[:, None] ** 2 + r[None, :] ** 2)) @ w), h, "cpu")
    ssm = (cfg.sqrts / (2 * MP + 2.1206)) ** 2
    sig = 0.1 * (34.41 + 0.2720 * math.log(ssm) ** 2 + 13.07 * ssm ** -0.4473 - 7.394 * ssm ** -0.5486)
    T = lambda x: ta(torch.from_numpy(np.minimum(x, 20.0))).numpy()
    phi = sum(2 * math.pi * wk * T(np.sqrt(np.maximum(
        r[:, None] ** 2 + r[None, :] ** 2 + 2 * r[:, None] * r[None, :] * math.cos(math.pi * x), 0.0)))
        for x, wk in zip(GLX, GLW))
    return _Spline(np.exp(-sig * ((2.0 * r * T(r))[None, :] * phi) @ w), h, dev)


def _exact_lumi(cfg, M, Y, scale):
    """L(M, Y) with the point-charge flux and no breakup factor, times scale."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    G = _overlap(cfg, dev)
    g = cfg.sqrts / (2 * MP)
    fac = cfg.Z ** 2 * ALPHA / math.pi ** 2 / HC ** 2

    def row(k):
        bmax = torch.clamp(5 * g * HC / k, min=5 * cfg.R)
        logd = (torch.log(bmax) - math.log(cfg.R)) / 120
        j = torch.arange(121, dtype=torch.float64, device=dev)
        e = cfg.R * torch.exp(logd[:, None] * j[None, :])
        b = (e[:, 1:] + e[:, :-1]) / 2
        x = b * k[:, None] / g / HC
        k0, k1 = torch.special.modified_bessel_k0(x), torch.special.modified_bessel_k1(x)
        return b, (fac * k / g / g)[:, None] * (k1 * k1 + k0 * k0 / g / g) * b * (e[:, 1:] - e[:, :-1])

    outs = []
    for c0 in range(0, M.numel(), 512):
        m, y = M[c0:c0 + 512].to(dev), Y[c0:c0 + 512].to(dev)
        b1, w1 = row(m / 2 * torch.exp(y))
        b2, w2 = row(m / 2 * torch.exp(-y))
        ww = w1[:, :, None] * w2[:, None, :]
        s = [0.0, 0.0]
        for x, wk in zip(GLX, GLW):
            co = math.cos(math.pi * x)
            d = b1[:, :, None] ** 2 + b2[:, None, :] ** 2 + (-2 if cfg.use_polarized else 2) * co * (
                b1[:, :, None] * b2[:, None, :])
            d = torch.sqrt(torch.clamp(d, min=0.0))
            v = (ww * torch.where(d < 20.0, G(torch.clamp(d, max=20.0)), torch.ones_like(d))).sum((1, 2)) * wk
            s[0] = s[0] + (v * co * co if cfg.use_polarized else v)
            s[1] = s[1] + v * math.sin(math.pi * x) ** 2
        pre = 2 * math.pi ** 2 * m * scale
        outs.append([(pre * v).cpu() for v in s[:1 + cfg.use_polarized]])
    res = tuple(torch.cat(v) for v in zip(*outs))
    return res if cfg.use_polarized else res[0]


def _philox(seed, ctr, sub):
    """Philox4x32-10 of (event, sub-block): two uniforms in [0, 1) of 53 bits."""
    mask = 0xFFFFFFFF
    c = [ctr & mask, ctr >> 32, torch.full_like(ctr, sub), torch.zeros_like(ctr)]
    k0, k1 = seed & mask, seed >> 32
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    u = lambda hi, lo: ((hi >> 5).double() * 67108864.0 + (lo >> 6).double()) * (1.0 / 9007199254740992.0)
    return u(c[0], c[1]), u(c[2], c[3])


def _exact_draws(case, seed):
    cfg = _config(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = {k: v.to(dev) for k, v in _tables(case, seed, cfg).items()}
    nm, ny, nz = case["nm"], case["ny"], case["nz"]
    outs = []
    for c0 in range(0, case["n"], 1 << 21):
        ctr = torch.arange(c0, min(case["n"], c0 + (1 << 21)), device=dev)
        r1, r2 = _philox(12345 + seed, ctr, 0)
        r3, r4 = _philox(12345 + seed, ctr, 1)
        k = torch.searchsorted(t["sum_ym"], r1, right=True) - 1
        iy, jm = (k // nm).double(), (k % nm).double()
        dy, dm = (cfg.ymax - cfg.ymin) / ny, (cfg.mmax - cfg.mmin) / nm
        y0, m0 = cfg.ymin + dy * iy, cfg.mmin + dm * jm
        y = y0 + (r1 - t["sum_ym"][k]) / (t["sum_ym"][k + 1] - t["sum_ym"][k]) * (cfg.ymin + dy * (iy + 1) - y0)
        m = m0 + r2 * (cfg.mmin + dm * (jm + 1) - m0)
        yb = ((ny * (y - cfg.ymin)).long().double() / (cfg.ymin + dy * ny - cfg.ymin)).long().clamp(max=ny - 1)
        mb = ((nm * (m - cfg.mmin)).long().double() / (cfg.mmin + dm * nm - cfg.mmin)).long().clamp(max=nm - 1)
        if case["pol"]:
            first = (r4 < t["ratio"][yb, mb])[:, None]
            rows = torch.where(first, t["sum_zs"][mb], t["sum_zp"][mb])
        else:
            rows = t["sum_z"][mb]
        zb = torch.searchsorted(rows, r3[:, None].contiguous(), right=True) - 1
        lo, hi = rows.gather(1, zb)[:, 0], rows.gather(1, zb + 1)[:, 0]
        zb, dz = zb[:, 0].double(), (cfg.zmax - cfg.zmin) / nz
        z0 = cfg.zmin + dz * zb
        z = z0 + (r3 - lo) / (hi - lo) * (cfg.zmin + dz * (zb + 1) - z0)
        outs.append((y.cpu(), m.cpu(), z.cpu()))
    return tuple(torch.cat(v) for v in zip(*outs))


def _exact_net(case, seed):
    nets, X, L0, T = _net(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    X, L0, T = (torch.from_numpy(v).to(dev).double() for v in (X, L0, T))

    def forward(p, x):
        ws, o = [], 0
        for s in NET_SHAPES:
            n = math.prod(s)
            ws.append(p[o:o + n].reshape(s))
            o += n
        for w, b in ((ws[0], ws[1]), (ws[2], ws[3]), (ws[4], ws[5])):
            x = torch.nn.functional.silu(x @ w.T + b)
        return x @ ws[6] + ws[7]

    ps = [torch.from_numpy(p).to(dev).double().requires_grad_(True) for p in nets]
    with torch.no_grad():
        r = [0.1 + 0.7 * forward(p, X[:case["infer"]]) for p in ps]
    grads = []
    for p in ps:
        ((forward(p, X[:case["rows"]]) - T[:case["rows"]]) ** 2).mean().backward()
        grads.append(p.grad.cpu())
    return (L0[:case["infer"]] + 0.5 * (r[0] + r[1])).cpu(), (r[0] - r[1]).abs().cpu(), grads[0], grads[1]


def _exact_zm(cfg):
    """dsigma/dz dM shape of gamma gamma -> l l (no anomalous moment) on the grid's lower edges, and its CDFs."""
    mass = {11: 0.000510998946, 13: 0.1056583745, 15: 1.77686}[cfg.proc_id]
    dm, dz = (cfg.mmax - cfg.mmin) / cfg.nm, (cfg.zmax - cfg.zmin) / cfg.nz
    m = cfg.mmin + dm * torch.arange(cfg.nm, dtype=torch.float64)[:, None]
    z = cfg.zmin + dz * torch.arange(cfg.nz, dtype=torch.float64)[None, :]
    k = m / 2
    p = torch.sqrt(k * k - mass * mass)
    kt, ku = -2 * k * (k - z * p) / mass ** 2, -2 * k * (k + z * p) / mass ** 2
    kq, kr = 1 / kt + 1 / ku, ku / kt + kt / ku
    zm = 2 * math.pi * ALPHA ** 2 / (m * m) * p / k * (-8.0 * (4 * kq * kq + 4 * kq - kr)) * (HC * HC * 1e7) / dm
    c = torch.cumsum(zm / zm.mean(1, keepdim=True) / cfg.nz, 1)
    return zm, torch.cat([torch.zeros(cfg.nm, 1, dtype=torch.float64), c], 1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("points", "grid"):
        # the form-factor flux is what an adaptive rule at 1e-4 makes of its integral, and the breakup
        # factor a table of data: neither has a value of its own
        npts = case["n"] if kind == "points" else case["nm"] * case["ny"]
        if not case["flux_point"] or case["mode"] != 1 or npts > 20000:
            return None
        cfg = _config(case, seed)
        if kind == "points":
            return _exact_lumi(cfg, *_points(case, seed), 1.0)
        dm, dy = (cfg.mmax - cfg.mmin) / cfg.nm, (cfg.ymax - cfg.ymin) / cfg.ny
        M = (cfg.mmin + dm * torch.arange(cfg.nm, dtype=torch.float64)).repeat_interleave(cfg.ny)
        Y = (cfg.ymin + dy * torch.arange(cfg.ny, dtype=torch.float64)).repeat(cfg.nm)
        L = _exact_lumi(cfg, M, Y, dm * dy)
        return tuple(v.reshape(cfg.nm, cfg.ny) for v in L) if cfg.use_polarized else L.reshape(cfg.nm, cfg.ny)
    if kind == "step":
        zm, sum_z = _exact_zm(_config(case, seed))
        return dict(zm=zm, sum_z=sum_z, L=None, cs=None, sum_ym=None, tot=None)
    if kind == "draws":
        return _exact_draws(case, seed)
    if kind == "net":
        pred, spread, g0, g1 = _exact_net(case, seed)
        return (pred, spread), g0, g1
    return None
