"""The work whose speed is measured: calls of the package's public entry points.

Each case is one call, or the few calls that a time step makes together, on
seeded inputs resident on the GPU.  The grids are latitude-longitude B-grids
with smooth random bathymetry, as mom5_amd.synth builds them: global domains
(cyclic in x, 10S to 80N) and closed regional basins.  Transports come from a
streamfunction plus an overturning with w from continuity, scaled to a largest
Courant number of 0.3; layer thicknesses follow a free surface.  Every pass
reads one time level and writes the other, so a pass can be repeated.

Sizes are those of the workloads of this repository (90x60x25 and 1440x1080x50
global grids, 3600x2700 eddying grids, 200-800 x 150-600 x 30-50 regional
basins, 75 levels), with an odd regional basin of 517x389x41.
"""
import math
import types

import numpy as np
import torch

from mom5_amd.ensemble import EnsembleStep
from mom5_amd.ocean import DeviceArray, OceanGPU
from mom5_amd.step import BatchedStep

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64, F32 = torch.float64, torch.float32

RADIUS, OMEGA, GRAV, RHO0 = 6371.0e3, 7.292e-5, 9.80, 1035.0
EPS40, EPS30 = 1.0e-40, 1.0e-30
GAMMA = 0.2                              # predictor weight of the barotropic
LIMITS = {"temp": (-2.0, 32.0), "salt": (1.0, 42.0), "passive": (-0.1, 1.0)}
MOST_WORK = 2400 * 1800 * 75 * 12        # tracer-cells of the largest tracer case


def listed():
    return [
        # the smallest whole step: a coarse global model (T, S, 80 subcycles)
        dict(name="coarse_step", kind="step", ni=90, nj=60, nk=25, cyclic=True, n64=2, n32=0,
             nts=80),
        # one regional basin with a biogeochemical set of passive tracers
        dict(name="regional_tracers", kind="tracers", ni=517, nj=389, nk=41, cyclic=False, n64=2,
             n32=6, quick=False, upwind=False, th=False),
        # a global quarter-degree model, every tracer in FP64
        dict(name="global_tracers_f64", kind="tracers", ni=1440, nj=1080, nk=50, cyclic=True,
             n64=8, n32=0, quick=False, upwind=False, th=False),
        # an eddying global model, T and S in FP64 and ten passive tracers in FP32
        dict(name="eddying_tracers_mixed", kind="tracers", ni=2400, nj=1800, nk=75, cyclic=True,
             n64=2, n32=10, quick=False, upwind=False, th=False),
        # T and S by the Quicker scheme, passive tracers by MDFL-Sweby
        dict(name="global_tracers_quicker", kind="tracers", ni=1440, nj=1080, nk=50, cyclic=True,
             n64=4, n32=0, quick=True, upwind=False, th=False),
        # one call per reference routine and tracer: T, S MDFL-Sweby, one Quicker
        dict(name="plain_tracers", kind="plain", ni=1440, nj=1080, nk=50, cyclic=True),
        # the split-explicit barotropic of an eddying global model
        dict(name="eddying_barotropic", kind="barotropic", ni=3600, nj=2700, cyclic=True, nts=120,
             cgrid=False, press=False),
        # ... of one regional basin
        dict(name="regional_barotropic", kind="barotropic", ni=517, nj=389, cyclic=False, nts=80,
             cgrid=False, press=False),
        # ... of a C-grid model in pressure coordinates
        dict(name="cgrid_press_barotropic", kind="barotropic", ni=1440, nj=1080, cyclic=True,
             nts=80, cgrid=True, press=True),
        # several uneven regional basins advanced together, whole steps
        dict(name="regional_ensemble", kind="ensemble", ndom=8, most=800, n32=6, nts=80),
        # advection velocity, barotropic forcing, surface height, closure
        dict(name="transports_closure", kind="transports", ni=1440, nj=1080, nk=50, cyclic=True,
             press=False),
        # implicit vertical diffusion with a neutral-physics K33 per tracer
        dict(name="neutral_diffusion", kind="diffusion", ni=1440, nj=1080, nk=50, cyclic=True,
             n64=3, k33=True),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "tracers", "tracers", "tracers", "plain", "barotropic",
                       "barotropic", "ensemble", "transports", "diffusion"])
    cyclic = rng.random() < 0.6
    ni = log(60, 3600) if cyclic else log(60, 800)
    nj = max(30, int(ni * rng.uniform(0.55, 0.8)))
    nk = rng.randint(20, 75)
    if kind == "ensemble":
        return dict(kind=kind, ndom=rng.randint(3, 8), most=rng.randint(300, 700),
                    n32=rng.randint(0, 6), nts=2 * rng.randint(20, 40))
    if kind == "barotropic":
        cgrid, press = rng.choice([(False, False), (False, False), (True, False), (False, True),
                                   (True, True)])
        if (cgrid or press) and ni > 1440:
            ni, nj = ni // 2, nj // 2
        return dict(kind=kind, ni=ni, nj=nj, cyclic=cyclic, nts=2 * rng.randint(20, 60),
                    cgrid=cgrid, press=press)
    quick = rng.random() < 0.35
    n64 = 2 + (rng.randint(0, 4) if rng.random() < 0.5 else 0)
    n32 = rng.choice([0, 0, 1, 3, 4, 6, 10])
    most = MOST_WORK * 0.9 / (n64 + n32) if kind == "tracers" else 1440 * 1080 * 50
    if kind == "step":
        most, n32 = min(most, MOST_WORK / 16), min(n32, 6)
    while ni * nj * nk > most or ni * nj * nk * (9 * 8 + 16 * n64 + 8 * n32) > 55e9:
        ni, nj = int(ni * 0.9), int(nj * 0.9)
    base = dict(kind=kind, ni=ni, nj=nj, nk=nk, cyclic=cyclic)
    if kind == "step":
        return dict(base, n64=n64, n32=n32, nts=2 * rng.randint(20, 60))
    if kind == "tracers":
        return dict(base, n64=n64, n32=n32, quick=quick, upwind=quick and rng.random() < 0.5,
                    th=rng.random() < 0.3)
    if kind == "transports":
        return dict(base, press=rng.random() < 0.5)
    if kind == "diffusion":
        return dict(base, n64=rng.randint(2, 4), k33=rng.random() < 0.5)
    return base


# ---- device arrays that are torch tensors ------------------------------------

class TensorArray(DeviceArray):
    """A field held by a torch tensor, as the package's entry points take it."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t, self.ptr = t, t.data_ptr()
        self.shape = tuple(t.shape)
        self.dtype = np.dtype({F64: np.float64, F32: np.float32, torch.int32: np.int32}[t.dtype])
        self.nbytes = t.numel() * t.element_size()

    def free(self):
        self.t = None


def arr(t):
    return None if t is None else TensorArray(t.contiguous())


# ---- inputs ------------------------------------------------------------------

class Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))
        self.rng = np.random.default_rng(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, dtype=F64, device=DEV, generator=self.g)

    def uniform(self, *shape):
        return torch.rand(*shape, dtype=F64, device=DEV, generator=self.g)

    def smooth(self, ni, nj, nmodes, kmax, cyclic):
        """A sum of random long waves on the compute domain (nj, ni)."""
        x = (torch.arange(ni, dtype=F64, device=DEV) + 0.5) / ni
        y = (torch.arange(nj, dtype=F64, device=DEV) + 0.5) / nj
        out = torch.zeros(nj, ni, dtype=F64, device=DEV)
        for _ in range(nmodes):
            kx = int(self.rng.integers(1, kmax + 1)) if cyclic else float(self.rng.uniform(0.5, kmax))
            ky = float(self.rng.uniform(0.5, kmax))
            p, q = self.rng.uniform(0, 2 * math.pi, 2)
            a = self.rng.uniform(0.5, 1.0) / (kx * kx + ky * ky) ** 0.5
            out += a * torch.outer(torch.cos(2 * math.pi * ky * y + q),
                                   torch.cos(2 * math.pi * kx * x + p))
        return out


def wrap(a, cyclic):
    """Halo columns as MOM's halo update leaves them (closed: land)."""
    if cyclic:
        a[..., 0] = a[..., -2]
        a[..., -1] = a[..., 1]
    else:
        a[..., 0] = 0
        a[..., -1] = 0
    return a


def embed(a, cyclic):
    """A compute-domain field on the data domain, land beyond closed edges."""
    out = torch.zeros(a.shape[:-2] + (a.shape[-2] + 2, a.shape[-1] + 2), dtype=a.dtype, device=DEV)
    out[..., 1:-1, 1:-1] = a
    return wrap(out, cyclic)


def make_grid(r, ni, nj, nk, cyclic, land=0.3):
    """Metrics, depths and masks (fields named as MOM's)."""
    NI, NJ = ni + 2, nj + 2
    if cyclic:
        lat_s, dlat, dlon = -10.0, 90.0 / nj, 360.0 / ni
    else:
        lat_s, dlat, dlon = -30.0, min(0.1, 100.0 / nj), 0.1
    jj = torch.arange(NJ, dtype=F64, device=DEV)
    lat_t = torch.deg2rad(lat_s + (jj - 0.5) * dlat)
    lat_u = torch.deg2rad(lat_s + jj * dlat)
    one = torch.ones(NJ, NI, dtype=F64, device=DEV)
    dlon_r, dlat_r = math.radians(dlon), math.radians(dlat)
    dxt = (RADIUS * torch.cos(lat_t) * dlon_r)[:, None] * one
    dxu = (RADIUS * torch.cos(lat_u).clamp_min(1e-3) * dlon_r)[:, None] * one
    dy = RADIUS * dlat_r * one
    G = types.SimpleNamespace(ni=ni, nj=nj, nk=nk, cyclic=cyclic, dxt=dxt, dyt=dy, dat=dxt * dy,
                              dxte=dxt, dyte=dy, dxtn=dxu, dytn=dy, dxu=dxu, dyu=dy)
    G.datr, G.dxur, G.dyur = 1.0 / (G.dat + EPS40), 1.0 / (dxu + EPS40), 1.0 / (dy + EPS40)
    G.f = (2.0 * OMEGA * torch.sin(lat_u))[:, None] * one
    ratio = (500.0 / 10.0) ** (1.0 / (nk - 1))
    dzt = 10.0 * ratio ** np.arange(nk)
    zw = np.cumsum(dzt)
    zt = zw - 0.5 * dzt
    dzw = np.concatenate([[zt[0]], zt[1:] - zt[:-1], [zw[-1] - zt[-1]]])
    G.dzt, G.zw, G.zt, G.dzw = (torch.as_tensor(a, dtype=F64, device=DEV) for a in (dzt, zw, zt, dzw))
    b = r.smooth(ni, nj, 12, 6, cyclic)
    q = torch.sort(b.flatten()[:: max(1, b.numel() // 1000000)])[0]
    q = q[int(land * (q.numel() - 1))]
    h = ((b - q) / (b.max() - q)).clamp(0.0, 1.0)
    depth = G.zw[-1] * (0.2 + 1.6 * h).clamp(0.0, 1.0)
    k = (torch.searchsorted(G.zw, depth * (1 - 1e-12)) + 1).clamp_max(nk)
    k[b <= q] = 0
    if not cyclic:
        k[:, 0] = 0
        k[:, -1] = 0
    kmt = embed(k.to(torch.int32), cyclic)
    kmu = torch.zeros_like(kmt)
    kmu[:-1, :-1] = torch.minimum(torch.minimum(kmt[:-1, :-1], kmt[:-1, 1:]),
                                  torch.minimum(kmt[1:, :-1], kmt[1:, 1:]))
    if cyclic:
        kmu[:, -1] = kmu[:, 1]
    G.kmt, G.kmu = kmt, kmu
    G.tmask1, G.umask1 = (kmt >= 1).to(F64), (kmu >= 1).to(F64)
    G.hu = torch.zeros(NJ, NI, dtype=F64, device=DEV)
    wet = kmu > 0
    G.hu[wet] = G.zw[(kmu[wet] - 1).long()]
    G.ht = torch.where(kmt > 0, G.zw[(kmt - 1).clamp_min(0).long()], torch.zeros_like(G.hu))
    cg = torch.sqrt(GRAV * G.hu.clamp_min(1.0))
    G.dtbt = max(1.0, math.floor(0.35 * float((torch.minimum(dxu, dy) / cg)[wet].min()) * 64)) / 64
    return G


def levels(G):
    return torch.arange(1, G.nk + 1, device=DEV, dtype=torch.int32)[:, None, None]


def domain(G):
    return dict(isd=0, ied=G.ni + 1, jsd=0, jed=G.nj + 1, isc=1, iec=G.ni, jsc=1, jec=G.nj,
                nk=G.nk, cyclic_x=int(G.cyclic), cyclic_y=0)


def context(G):
    names = ("dxt", "dyt", "dat", "datr", "dxte", "dyte", "dxtn", "dytn", "dxu", "dyu", "dxur",
             "dyur", "f", "kmt", "kmu", "dzt")
    keep = {n: arr(getattr(G, n)) for n in names}
    torch.cuda.synchronize()
    return OceanGPU(domain(G), keep)


def faces_u(G, tm):
    """1 on the east (north) faces between two wet cells."""
    e, n = torch.zeros_like(tm), torch.zeros_like(tm)
    e[..., :-1] = tm[..., :-1] * tm[..., 1:]
    n[:, :-1] = tm[:, :-1] * tm[:, 1:]
    e[:, 0], e[:, -1], n[:, -1] = 0, 0, 0
    return e, n


def make_flow(G, r, nts):
    """Transports and wrho_bt by continuity, rho_dzt, and the time step."""
    nk, cyc = G.nk, G.cyclic
    tm = (levels(G) <= G.kmt).to(F64)
    thick = 1.0 + embed(0.3 * r.smooth(G.ni, G.nj, 6, 5, cyc), cyc) / 3000.0
    rho = RHO0 * G.dzt[:, None, None] * thick
    # horizontal streamfunction on U points, decaying with depth
    psi = embed(r.smooth(G.ni, G.nj, 8, 4, cyc), cyc)
    psik = psi * torch.exp(-G.zt / 1000.0)[:, None, None] * (levels(G) <= G.kmu).to(F64)
    coef = (RHO0 * G.dzt)[:, None, None]
    mx, my = torch.zeros_like(tm), torch.zeros_like(tm)
    mx[:, 1:] = coef * (psik[:, 1:] - psik[:, :-1])
    my[:, :, 1:] = -coef * (psik[:, :, 1:] - psik[:, :, :-1])
    del psik
    # an x-z overturning without a vertical integral
    ov = embed(r.smooth(G.ni, G.nj, 6, 3, cyc), cyc)
    kf = torch.zeros_like(G.kmt)
    kf[:, :-1] = torch.minimum(G.kmt[:, :-1], G.kmt[:, 1:])
    if cyc:
        kf[:, -1] = kf[:, 1]
    hf = torch.where(kf > 0, G.zw[(kf - 1).clamp_min(0).long()], torch.ones_like(ov))
    amp = 0.3 * float(mx.abs().max()) / (RHO0 * float(ov.abs().max()))
    up = torch.zeros_like(ov)
    for k in range(nk):
        dn = torch.where(k + 1 < kf, ov * torch.sin(math.pi * G.zw[k] / hf.clamp_min(1.0)),
                         torch.zeros_like(ov))
        mx[k] += RHO0 * amp * (up - dn)
        up = dn
    e, n = faces_u(G, tm)
    mx *= e
    my *= n
    del e, n
    wrap(mx, cyc)
    wrap(my, cyc)
    w = torch.zeros(nk + 1, *tm.shape[1:], dtype=F64, device=DEV)
    for k in range(nk):
        div = torch.zeros_like(ov)
        div[:, 1:] += mx[k, :, 1:] - mx[k, :, :-1]
        div[1:] += my[k, 1:] - my[k, :-1]
        w[k + 1] = (div * G.datr + w[k]) * tm[k]
    w[:, 0] = 0.0
    w[:, -1] = 0.0
    wrap(w, cyc)
    dt = G.dtbt * nts / 2.0
    cx = (mx[:, :, :-1] / (G.dyte * G.dxte)[:, :-1] * 2.0 / (rho[:, :, :-1] + rho[:, :, 1:])).abs().max()
    cy = (my[:, :-1] / (G.dxtn * G.dytn)[:-1] * 2.0 / (rho[:, :-1] + rho[:, 1:])).abs().max()
    cz = (w[1:] / rho).abs().max()
    s = 0.3 / (dt * max(float(cx), float(cy), float(cz)))
    mx *= s / G.dyte
    my *= s / G.dxtn
    w *= s
    out = thick * (1.0 + 1e-5 * embed(r.smooth(G.ni, G.nj, 4, 5, cyc), cyc))
    return types.SimpleNamespace(u=mx, v=my, w=w, rho=rho, dt=dt,
                                 rhor=1.0 / (RHO0 * G.dzt[:, None, None] * out + EPS40),
                                 dzwt=(G.dzw[:, None, None] * thick).contiguous())


def make_tracer(G, r, kind, dtype=F64):
    n = r.normal(G.nk, G.nj, G.ni)
    if kind == "temp":
        n.mul_(0.5).add_((2.0 + 25.0 * torch.exp(-G.zt / 800.0))[:, None, None])
    elif kind == "salt":
        n.mul_(0.2).add_(35.0)
    else:
        n.mul_(1.5).add_(math.log(1e-3)).exp_()
    n *= (levels(G) <= G.kmt[1:-1, 1:-1])
    return embed(n.to(dtype), G.cyclic)


def make_mixing(G, r):
    d = torch.zeros(2, G.nk, G.nj + 2, G.ni + 2, dtype=F64, device=DEV)
    for p in range(2):
        d[p, :, 1:-1, 1:-1] = 10.0 ** (-5.0 + 3.0 * r.uniform(G.nk, G.nj, G.ni))
    return wrap(d, G.cyclic)


def make_surface(G, r, scale, mask=None):
    return embed(scale * r.normal(G.nj, G.ni), G.cyclic) * (G.tmask1 if mask is None else mask)


def kinds_of(c):
    return (["temp", "salt"] + ["passive"] * (c.get("n64", 3) + c.get("n32", 0) - 2))


def make_bt(G, r, cgrid=False, press=False):
    """State and 2-D inputs of the barotropic subcycle."""
    B = types.SimpleNamespace()
    if cgrid:
        m = torch.zeros(2, *G.tmask1.shape, dtype=F64, device=DEV)
        m[0, :-1, :-1] = torch.minimum(G.tmask1[:-1, :-1], G.tmask1[:-1, 1:])
        m[1, :-1, :-1] = torch.minimum(G.tmask1[:-1, :-1], G.tmask1[1:, :-1])
        if G.cyclic:
            m[:, 1:-1, 0], m[:, 1:-1, -1] = m[:, 1:-1, -2], m[:, 1:-1, 1]
        B.tmasken = m
    else:
        B.tmasken, m = None, torch.stack([G.umask1, G.umask1])
    scale = RHO0 * GRAV if press else 1.0
    B.x = scale * make_surface(G, r, 0.1)
    B.ud = torch.stack([make_surface(G, r, 30.0, m[c]) for c in range(2)])
    B.forcing = torch.stack([make_surface(G, r, 0.3, m[c]) for c in range(2)])
    if cgrid:
        B.thick = torch.stack([torch.minimum(G.ht, G.ht.roll(-1, 1)) * m[0],
                               torch.minimum(G.ht, G.ht.roll(-1, 0)) * m[1]])
        wrap(B.thick, G.cyclic)
    else:
        B.thick = G.hu.clone()
    if press:
        B.thick = RHO0 * B.thick
    one = torch.ones_like(G.tmask1)
    B.patm = 1.0e5 + make_surface(G, r, 200.0, one)
    B.rho_g = GRAV * (1025.0 + make_surface(G, r, 2.0, one))
    B.dpatm_dt = make_surface(G, r, 1e-3, one)
    B.pme, B.river = make_surface(G, r, 5e-5), make_surface(G, r, 1e-5).abs()
    B.source = torch.zeros_like(one)
    B.smooth = make_surface(G, r, 1e-6)
    return B


def regional_sizes(c, seed=4):
    """The uneven basins of an ensemble (200-800 x 150-600 x 30-50 at full size)."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(c["ndom"]):
        ni = int(rng.integers(c["most"] // 4, c["most"] + 1))
        nj = int(rng.integers(c["most"] * 3 // 16, c["most"] * 3 // 4 + 1))
        nts = max(20, int(rng.integers(c["nts"] // 2, c["nts"] * 3 // 2)) // 2 * 2)
        out.append((ni, nj, int(rng.integers(30, 51)), nts))
    return out


def inputs(case, seed):
    """What prepare() puts on the GPU and exact() computes from."""
    r = Rand(seed)
    if case["kind"] == "ensemble":
        return [inputs(dict(kind="step", ni=ni, nj=nj, nk=nk, cyclic=False, n64=2, n32=case["n32"],
                            nts=nts), seed * 64 + k)
                for k, (ni, nj, nk, nts) in enumerate(regional_sizes(case))]
    kind = case["kind"]
    G = make_grid(r, case["ni"], case["nj"], case.get("nk", 25), case["cyclic"])
    I = types.SimpleNamespace(G=G)
    if kind in ("step", "tracers", "plain"):
        I.flow = make_flow(G, r, case.get("nts", 80))
        n64 = case.get("n64", 3)
        I.kinds = kinds_of(case)
        I.T = [make_tracer(G, r, k, F64 if n < n64 else F32) for n, k in enumerate(I.kinds)]
        I.mix = make_mixing(G, r)
    if kind in ("step", "tracers", "plain", "diffusion"):
        n = len(kinds_of(case))
        if kind == "diffusion":
            thick = 1.0 + embed(0.3 * r.smooth(G.ni, G.nj, 6, 5, G.cyclic), G.cyclic) / 3000.0
            I.flow = types.SimpleNamespace(rho=RHO0 * G.dzt[:, None, None] * thick, dt=1800.0,
                                           dzwt=(G.dzw[:, None, None] * thick).contiguous())
            I.kinds = kinds_of(case)
            I.T = [make_tracer(G, r, k) for k in I.kinds]
            I.mix = make_mixing(G, r)
            I.k33 = ([embed(10.0 ** (-2.0 + 3.0 * r.uniform(G.nk, G.nj, G.ni)), G.cyclic)
                      for _ in range(n)] if case["k33"] else None)
        I.stf = [make_surface(G, r, 1e-4) for _ in range(n)]
        I.btf = [make_surface(G, r, 1e-6) for _ in range(n)]
    I.nts = case.get("nts")
    I.th = None
    if case.get("th"):
        I.th = [embed(1e-4 * r.normal(G.nk, G.nj, G.ni), G.cyclic)
                * (levels(G) <= G.kmt) for _ in I.kinds]
    if kind in ("step", "barotropic"):
        I.bt = make_bt(G, r, case.get("cgrid", False), case.get("press", False))
    if kind == "transports":
        um = (levels(G) <= G.kmu).to(F64)
        I.u = torch.stack([embed(0.2 * r.normal(G.nk, G.nj, G.ni), G.cyclic) * um for _ in range(2)])
        I.rho_dzu = (RHO0 * G.dzt[:, None, None]
                     * (1.0 + embed(1e-4 * r.normal(G.nj, G.ni), G.cyclic))).contiguous()
        I.tend = embed(1e-5 * r.normal(G.nk, G.nj, G.ni), G.cyclic)
        I.accel = torch.stack([embed(1e-3 * r.normal(G.nk, G.nj, G.ni), G.cyclic) for _ in range(2)])
        I.smf = torch.stack([make_surface(G, r, 0.1, G.umask1) for _ in range(2)])
        I.bmf = torch.stack([make_surface(G, r, 0.01, G.umask1) for _ in range(2)])
        I.bt = make_bt(G, r, False, case["press"])
        I.conv = make_surface(G, r, 1e-3)
        I.anompb = make_surface(G, r, 1.0e3)
        half = (0.5 * G.dxt, 0.5 * G.dxt, 0.5 * G.dyt, 0.5 * G.dyt)
        I.remap = [a.clone() for a in half] + [1.0 / (G.dxu * G.dyu)]
    return I


# ---- one pass ------------------------------------------------------------------

def zeros_like(t):
    return torch.zeros_like(t)


def tracer_args(I, S, case):
    names = I.kinds
    quick = case.get("quick", False)
    kw = dict(uhrho_et=S.u, vhrho_nt=S.v, wrho_bt=S.w, rho_dzt_tau=S.rho, rho_dztr=S.rhor,
              dtime=I.flow.dt, stfs=S.stf, btfs=S.btf, dzwt=S.dzwt, diff_cbt=S.mix, index_salt=1,
              th_tendencies=S.th)
    if quick:
        kw.update(schemes=["quicker" if n < 2 else "mdfl_sweby" for n in range(len(names))],
                  min_limits=[LIMITS[k][0] for k in names],
                  max_limits=[LIMITS[k][1] for k in names], index_temp=0, ts_same=True,
                  limit_with_upwind=case.get("upwind", False))
    return kw


def prepare(case, seed):
    kind = case["kind"]
    I = inputs(case, seed)
    if kind == "ensemble":
        return prepare_ensemble(case, I)
    G, S = I.G, types.SimpleNamespace()
    S.kind, S.case, S.G = kind, case, G
    if kind in ("step", "tracers", "plain", "diffusion"):
        fl = I.flow
        S.dt, S.kinds, S.mix = fl.dt, I.kinds, arr(I.mix)
        S.T = [arr(t) for t in I.T]
        S.stf, S.btf = [arr(t) for t in I.stf], [arr(t) for t in I.btf]
        S.rho, S.dzwt = arr(fl.rho), arr(fl.dzwt)
        S.th = None if I.th is None else [arr(t) for t in I.th]
        if kind != "diffusion":
            S.u, S.v, S.w, S.rhor = arr(fl.u), arr(fl.v), arr(fl.w), arr(fl.rhor)
            S.out = [arr(zeros_like(t)) for t in I.T]
        else:
            S.k33 = None if I.k33 is None else [arr(t) for t in I.k33]
        if kind == "plain":
            S.tend = arr(torch.zeros_like(fl.rho))
            S.lim = [arr(torch.zeros_like(fl.rho)) for _ in I.T]
        elif kind != "diffusion":
            S.args = tracer_args(I, S, case)
    if kind in ("step", "barotropic"):
        S.bt, S.bt_out = bt_args(I, case)
    if kind == "transports":
        for n in ("u", "rho_dzu", "tend", "accel", "smf", "bmf", "conv", "anompb"):
            setattr(S, n, arr(getattr(I, n)))
        B = I.bt
        for n in ("pme", "river", "source", "patm", "rho_g", "dpatm_dt", "x"):
            setattr(S, n, arr(getattr(B, n)))
        S.ht = arr(G.ht)
        n3, n2 = torch.zeros_like(I.tend), torch.zeros_like(B.pme)
        S.o3 = [arr(zeros_like(n3)) for _ in range(3)]
        S.ow = arr(torch.zeros(G.nk + 1, *n2.shape, dtype=F64, device=DEV))
        S.o2 = {n: arr(zeros_like(n2)) for n in ("xp", "td", "pb", "eu", "ps")}
        S.o22 = {n: arr(torch.stack([n2, n2])) for n in ("fb", "gp", "ga")}
    S.gpu = context(G)
    if kind == "transports":
        S.gpu.set_remap_metrics(*[a.cpu().numpy() for a in I.remap])
    return S


def bt_args(I, case):
    B, G = I.bt, I.G
    cgrid, press = case.get("cgrid", False), case.get("press", False)
    out = [arr(zeros_like(B.x)), arr(zeros_like(B.ud)), arr(zeros_like(B.x))]
    kw = dict(nts=case["nts"], dtbt=G.dtbt, udrho_tau=arr(B.ud), forcing_bt=arr(B.forcing),
              pme=arr(B.pme), river=arr(B.river), source=arr(B.source), udrho_taup1=out[1],
              conv_rho_ud_t=out[2], pred_corr_gamma=GAMMA, rho0=RHO0)
    if not (cgrid or press):
        kw.update(eta_t_bar_tau=arr(B.x), thicku=arr(B.thick), patm=arr(B.patm),
                  eta_smooth=arr(B.smooth), rho_g=arr(B.rho_g), eta_t_bar_taup1=out[0])
    else:
        kw.update(cgrid=cgrid, pressure_based=press, x_bar_tau=arr(B.x), thick=arr(B.thick),
                  smooth=arr(B.smooth), x_bar_taup1=out[0], tmasken=arr(B.tmasken),
                  patm=arr(B.patm), rho_g=arr(B.rho_g), dpatm_dt=arr(B.dpatm_dt), grav=GRAV)
    return kw, out


def prepare_ensemble(case, parts):
    """Each member's outputs lie in arrays that all members share."""
    def flat(ts, dtype):
        return torch.zeros(sum(t.numel() for t in ts), dtype=dtype, device=DEV)

    S = types.SimpleNamespace(kind="ensemble", case=case)
    n32 = case["n32"]
    S.o64 = flat([t for I in parts for t in I.T[:2]], F64)
    S.o32 = flat([t for I in parts for t in I.T[2:]] or [torch.zeros(1)], F32)
    S.oeta = flat([I.bt.x for I in parts], F64)
    S.oud = flat([I.bt.ud for I in parts], F64)
    at = dict.fromkeys(("o64", "o32", "oeta", "oud"), 0)

    def cut(name, like):
        a, n = at[name], like.numel()
        at[name] = a + n
        return arr(getattr(S, name)[a:a + n].view(like.shape))

    members = []
    for I in parts:
        G, fl, B = I.G, I.flow, I.bt
        fields = dict(uhrho_et=fl.u, vhrho_nt=fl.v, wrho_bt=fl.w, rho_dzt=fl.rho, rho_dztr=fl.rhor,
                      dzwt=fl.dzwt, diff_cbt=I.mix, eta_t_bar=B.x, udrho=B.ud,
                      forcing_bt=B.forcing, thicku=B.thick, patm=B.patm, pme=B.pme, river=B.river,
                      source=B.source, eta_smooth=B.smooth, rho_g=B.rho_g)
        fields = {k: arr(v) for k, v in fields.items()}
        fields.update(stf=[arr(t) for t in I.stf], btf=[arr(t) for t in I.btf])
        names = ["temp", "salt"] + ["passive%02d" % n for n in range(n32)]
        gpu = context(G)
        c = types.SimpleNamespace(ni=G.ni, nj=G.nj, nk=G.nk, dom=domain(G), dt=fl.dt, dtbt=G.dtbt,
                                  nts=I.nts, fields=fields, grid=None,
                                  tracers=[(n, arr(t)) for n, t in zip(names, I.T)])
        m = BatchedStep(c, gpu=gpu)
        for n, t in enumerate(I.T):
            m.T[n][1] = cut("o64" if n < 2 else "o32", t)
        m.eta_bar[1], m.udrho[1] = cut("oeta", B.x), cut("oud", B.ud)
        members.append(m)
    S.ens = EnsembleStep(members)
    torch.cuda.synchronize()
    return S


def run(S):
    g = None if S.kind == "ensemble" else S.gpu
    if S.kind == "ensemble":
        S.ens.run()
        for m in S.ens.members:              # the next pass starts from the same time level
            m.cur = 0
        return [S.o64, S.o32, S.oeta, S.oud]
    if S.kind in ("tracers", "step"):
        g.step_tracers(S.T, S.out, **S.args)
        if S.kind == "tracers":
            return [a.t for a in S.out]
        g.update_ocean_barotropic(**S.bt)
        return [a.t for a in S.out + S.bt_out]
    if S.kind == "barotropic":
        if S.case["cgrid"] or S.case["press"]:
            g.update_ocean_barotropic_variant(**S.bt)
        else:
            g.update_ocean_barotropic(**S.bt)
        return [a.t for a in S.bt_out]
    if S.kind == "plain":
        g.compute_tmask_limit(S.T, [LIMITS[k][0] for k in S.kinds], [LIMITS[k][1] for k in S.kinds],
                              S.lim)
        for n, T in enumerate(S.T):
            scheme = "mdfl_sweby" if n < 2 else "quicker"
            g.fill(S.tend, 0.0)
            g.horz_advect_tracer(scheme, T, S.tend, uhrho_et=S.u, vhrho_nt=S.v, wrho_bt=S.w,
                                 rho_dzt_tau=S.rho, T_tau=T, dtime=S.dt, tmask_limit=S.lim[n])
            g.vert_advect_tracer(scheme, T, S.tend, wrho_bt=S.w, T_tau=T, tmask_limit=S.lim[n])
            g.update_tracer_explicit(T, S.tend, S.rho, S.rhor, S.dt, S.out[n])
        g.vert_diffuse_implicit(S.out, S.stf, S.btf, S.mix, S.rho, S.dzwt, S.dt)
        for t in S.out:
            g.update_domains(t)
        return [a.t for a in S.out + S.lim]
    if S.kind == "diffusion":
        g.vert_diffuse_implicit(S.T, S.stf, S.btf, S.mix, S.rho, S.dzwt, S.dt, K33s=S.k33)
        return [a.t for a in S.T]
    press = S.case["press"]
    o2, o22 = S.o2, S.o22
    g.advection_velocity(S.u, S.rho_dzu, S.pme, S.river, S.o3[0], S.o3[1], S.ow,
                         rho_dzt_tendency=S.tend, diverge_t=S.o3[2])
    g.barotropic_forcing(S.accel, S.smf, S.bmf, o22["fb"])
    g.eta_and_pbot_update(S.x, o2["xp"], o2["td"], conv_rho_ud_t_tau=S.conv, pme=S.pme,
                          river=S.river, source=S.source, dtime=1800.0, pressure_based=press,
                          dpatm_dt=S.dpatm_dt if press else None, ht=S.ht if press else None,
                          pbot_t_taup1=o2["pb"] if press else None)
    g.barotropic_closure(S.x, S.patm, S.rho_g, o2["eu"], o2["ps"], o22["gp"],
                         anompb_bar=S.anompb if press else None,
                         grad_anompb=o22["ga"] if press else None, pressure_based=press,
                         ht=S.ht if press else None)
    return ([a.t for a in S.o3] + [S.ow.t] + [a.t for a in o2.values()]
            + [a.t for a in o22.values()])


# ---- bytes and operations that a pass cannot do without -------------------------

def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        ws = [work(dict(kind="step", ni=ni, nj=nj, nk=nk, n64=2, n32=case["n32"], nts=nts))
              for ni, nj, nk, nts in regional_sizes(case)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    c2 = case["ni"] * case["nj"]
    c3 = c2 * case.get("nk", 1)
    n64, n32 = case.get("n64", 3), case.get("n32", 0)
    n = n64 + n32
    by = fl = 0.0
    if kind in ("step", "tracers", "plain"):
        # tracers read and written once; u, v, w, rho_dzt, 1/rho_dzt, dzwt and
        # two mixing planes; plain: the limits written too
        by += c3 * (16 * n64 + 8 * n32 + 64) + c2 * (52 + 16 * n)
        fl += c3 * (120.0 * n + 60)
        if kind == "plain":
            by += c3 * 8 * n
        if case.get("th"):
            by += c3 * 8 * n
    if kind == "diffusion":
        by += c3 * (16 * n64 + 32 + (8 * n64 if case["k33"] else 0)) + c2 * 16 * n64
        fl += c3 * 30.0 * n64
    if kind in ("step", "barotropic"):
        by += c2 * 156.0
        fl += c2 * 75.0 * case["nts"]
    if kind == "transports":
        by += c3 * 8.0 * (2 + 1 + 1 + 4 + 2) + c2 * 8.0 * 40
        fl += c3 * 40.0
    return {"bytes": float(by), "flops": float(fl)}


# ---- the same results in plain torch, FP64 ---------------------------------------

def pad(a, cyclic, n=2):
    """A compute-domain field with n more points a side: cyclic in x or zero, zero in y."""
    z = torch.zeros(a.shape[:-2] + (a.shape[-2] + 2 * n, a.shape[-1] + 2 * n), dtype=a.dtype,
                    device=a.device)
    z[..., n:-n, n:-n] = a
    if cyclic:
        z[..., n:-n, :n] = a[..., -n:]
        z[..., n:-n, -n:] = a[..., :n]
    return z


def flux(Rjm, Rj, Rjp, Tp, Tm, M, c, mm):
    d0 = (2.0 - c) * (1.0 - c) / 6.0
    d1 = (1.0 - c * c) / 6.0
    kk = (1.0 - c) / (EPS30 + c)

    def psi(R):
        th = R / (EPS30 + Rj)
        return torch.minimum((d0 + d1 * th).clamp_max(1.0), kk * th).clamp_min(0.0)

    return torch.where(M >= 0, M * (Tp + psi(Rjm) * Rj), M * (Tm - psi(Rjp) * Rj)) * mm


def ex_mdfl(T, fl, G):
    """The MDFL-Sweby th_tendency on the compute domain."""
    cyc, dt = G.cyclic, fl.dt
    c = (slice(None), slice(1, -1), slice(1, -1))
    T = T[c].to(F64)
    rho, w = fl.rho[c], fl.w[1:][c]
    dat, datr = G.dat[1:-1, 1:-1], G.datr[1:-1, 1:-1]
    m = (levels(G) <= G.kmt[1:-1, 1:-1]).to(F64)

    def k(a, s):
        return a[(torch.arange(G.nk, device=a.device) + s).clamp(0, G.nk - 1)]

    tp, mp = k(T, 1), k(m, 1)
    fb = flux((tp - k(T, 2)) * mp * k(m, 2), (T - tp) * m * mp, (k(T, -1) - T) * k(m, -1) * m,
              tp, T, dat * w, (w * dt / rho).abs(), m * mp)
    wm = torch.cat([torch.zeros_like(w[:1]), w[:-1]])
    ft = torch.cat([torch.zeros_like(w[:1]), fb[:-1]])
    tr = T + dt / rho * (datr * (fb - ft) + T * (wm - w))
    del fb, ft, tp, mp
    # x
    P, Q = pad(tr, cyc)[:, 2:-2], pad(m, cyc)[:, 2:-2]
    D = (P[..., 1:] - P[..., :-1]) * Q[..., 1:] * Q[..., :-1]
    u, dy = fl.u[:, 1:-1, :-1], G.dyte[1:-1, :-1]
    cf = (u * dt * 2.0 / ((fl.rho[:, 1:-1, :-1] + fl.rho[:, 1:-1, 1:]) * G.dxte[1:-1, :-1])).abs()
    fx = flux(D[..., :-2], D[..., 1:-1], D[..., 2:], P[..., 1:-2], P[..., 2:-1], dy * u, cf,
              Q[..., 1:-2] * Q[..., 2:-1])
    mu = dy * u
    tr = tr + dt * m * datr / rho * (fx[..., :-1] - fx[..., 1:] + T * (mu[..., 1:] - mu[..., :-1]))
    brk = w - wm + datr * (mu[..., :-1] - mu[..., 1:])
    del P, D, fx, cf, mu
    # y
    P, Q = pad(tr, cyc)[..., 2:-2], pad(m, cyc)[..., 2:-2]
    D = (P[:, 1:] - P[:, :-1]) * Q[:, 1:] * Q[:, :-1]
    v, dx = fl.v[:, :-1, 1:-1], G.dxtn[:-1, 1:-1]
    cf = (v * dt * 2.0 / ((fl.rho[:, :-1, 1:-1] + fl.rho[:, 1:, 1:-1]) * G.dytn[:-1, 1:-1])).abs()
    fy = flux(D[:, :-2], D[:, 1:-1], D[:, 2:], P[:, 1:-2], P[:, 2:-1], dx * v, cf,
              Q[:, 1:-2] * Q[:, 2:-1])
    tr = tr + dt * m * datr / rho * (fy[:, :-1] - fy[:, 1:])
    tr = tr + dt * T / rho * brk
    return rho * (tr - T) / dt * m


def ex_limit(T, lo, hi, G):
    """tmask_limit on (isc-1:iec, jsc-1:jec), from halo-updated T."""
    m = levels(G) <= G.kmt
    out = m & ((T < lo) | (T > hi))
    L = out[:, :-1, :-1] | out[:, :-1, 1:] | out[:, 1:, :-1]
    L[:-1] |= out[1:, :-1, :-1]
    return (L & m[:, :-1, :-1])


def quick_weights(x, d):
    """Quicker weights of the faces between cells d of a padded (2) axis."""
    n = x.shape[d]
    xm, x0, x1, x2 = (x.narrow(d, s, n - 3) for s in range(4))
    return ((x1 / (x1 + x0), x0 / (x1 + x0)),
            (x0 * x1 / ((xm + 2 * x0 + x1) * (x0 + x1)), -x0 * x1 / ((x0 + x1) * (xm + x0)),
             x0 * x1 / ((xm + 2 * x0 + x1) * (xm + x0))),
            (x0 * x1 / ((x0 + 2 * x1 + x2) * (x1 + x2)), -x0 * x1 / ((x1 + x2) * (x0 + x1)),
             x0 * x1 / ((x0 + 2 * x1 + x2) * (x0 + x1))))


def quick_flux(vel, P, Q, d, W):
    n = P.shape[d]
    tm, t0, t1, t2 = (P.narrow(d, s, n - 3) for s in range(4))
    mm, m0, m1, m2 = (Q.narrow(d, s, n - 3) for s in range(4))
    q, p, e = W
    a, b = m0 * (1.0 - mm), m1 * (1.0 - m2)
    return (vel * (q[0] * t0 + q[1] * t1)
            - vel.clamp_min(0) * (p[0] * t1 + p[1] * t0 + p[2] * (tm * (1 - a) + t0 * a))
            - vel.clamp_max(0) * (e[0] * (t2 * (1 - b) + t1 * b) + e[1] * t1 + e[2] * t0))


def ex_quicker(T, L, fl, G, upwind):
    """The Quicker th_tendency on the compute domain; L as ex_limit gives it."""
    cyc, nk = G.cyclic, G.nk
    m = (levels(G) <= G.kmt[1:-1, 1:-1]).to(F64)
    Tc = T[:, 1:-1, 1:-1]
    datr = G.datr[1:-1, 1:-1]

    def widths(a, d):
        a = a[1:-1, 1:-1]
        if d == 1 and cyc:
            return torch.cat([a[:, -2:], a, a[:, :2]], 1)
        return torch.cat([a.narrow(d, 0, 1)] * 2 + [a] + [a.narrow(d, a.shape[d] - 1, 1)] * 2, d)

    P, Q = pad(Tc, cyc), pad(m, cyc)
    Px, Qx, Py, Qy = P[:, 2:-2], Q[:, 2:-2], P[..., 2:-2], Q[..., 2:-2]
    u, v = fl.u[:, 1:-1, :-1], fl.v[:, :-1, 1:-1]
    dy, dx = G.dyte[1:-1, :-1], G.dxtn[:-1, 1:-1]
    fx = quick_flux(dy * u, Px, Qx, 2, quick_weights(widths(G.dxt, 1), 1))
    fy = quick_flux(dx * v, Py, Qy, 1, quick_weights(widths(G.dyt, 0), 0))
    if upwind:
        lx, ly = L[:, 1:], L[:, :, 1:]
        up = dy * (u.clamp_min(0) * Px[..., 1:-2] + u.clamp_max(0) * Px[..., 2:-1])
        fx = torch.where(lx, up * Qx[..., 1:-2] * Qx[..., 2:-1], fx)
        up = dx * (v.clamp_min(0) * Py[:, 1:-2] + v.clamp_max(0) * Py[:, 2:-1])
        fy = torch.where(ly, up * Qy[:, 1:-2] * Qy[:, 2:-1], fy)
    th = -m * (fx[..., 1:] - fx[..., :-1] + fy[:, 1:] - fy[:, :-1]) * datr
    Lc = L[:, 1:, 1:]
    z = torch.cat([G.dzt[:1], G.dzt, G.dzt[-1:], G.dzt[-1:]])
    q, p, e = quick_weights(z, 0)
    ft = torch.zeros_like(datr)
    for k in range(nk):
        km, kp, k2 = max(k - 1, 0), min(k + 1, nk - 1), min(k + 2, nk - 1)
        w = fl.w[k + 1, 1:-1, 1:-1]
        wn, wp = w.clamp_max(0), w.clamp_min(0)
        t2 = torch.where(m[k2] > 0, Tc[k2], Tc[kp])
        a = m[k] * (1.0 - m[km])
        f = (w * (q[0][k] * Tc[k] + q[1][k] * Tc[kp])
             - wn * (p[0][k] * Tc[kp] + p[1][k] * Tc[k] + p[2][k] * Tc[km])
             - wp * (e[0][k] * t2 + e[1][k] * Tc[kp] + e[2][k] * (Tc[k] * (1 - a) + Tc[kp] * a)))
        f = torch.where(Lc[k], (wn * Tc[k] + wp * Tc[kp]) * m[k] * m[kp], f)
        th[k] -= m[k] * (ft - f)
        ft = f
    return th


def ex_vdiff(T, stf, btf, dc, k33, fl, G):
    """The implicit vertical diffusion of T (data domain), in place."""
    c = (slice(1, -1), slice(1, -1))
    kmt, nk, dt = G.kmt[c], G.nk, fl.dt
    kb = kmt.clamp_min(2)
    E, z = [], []
    cp = bet = zp = None
    for k in range(1, nk + 1):
        def dcb(q):
            return RHO0 * dc[q - 1][c] + (0.0 if k33 is None else k33[q - 1][c])
        dh = fl.rho[k - 1][c]
        m, mn = (kmt >= k).to(F64), (kmt >= min(k + 1, nk)).to(F64)
        a = -dcb(max(k - 1, 1)) * dt / (fl.dzwt[k - 1][c] * dh) * m if k > 1 else torch.zeros_like(dh)
        cc = -dcb(k) * dt / (fl.dzwt[k][c] * dh) * mn if k < nk else torch.zeros_like(dh)
        b = 1.0 - a - cc
        f = T[k - 1][c] * (1.0 if k == 1 else m)
        if k == 1:
            f = f + stf[c] * dt * m / dh
            bet = m / (b + EPS30)
            zk = f * bet
            E.append(None)
        else:
            f = torch.where(kb == k, T[k - 1][c] - btf[c] * dt * m / dh, f)
            e = cp * bet
            bet = m / (b - a * e + EPS30)
            zk = (f - a * zp) * bet
            E.append(e)
        z.append(zk)
        cp, zp = cc, zk
    T[nk - 1][c] = z[-1]
    for k in range(nk - 1, 0, -1):
        z[k - 1] = z[k - 1] - E[k] * z[k]
        T[k - 1][c] = z[k - 1]
    return T


def ex_tracers(I, case):
    G, fl, outs, limits = I.G, I.flow, [], None
    quick = [False] * len(I.T)
    if case["kind"] == "plain":
        quick[2:] = [True] * (len(quick) - 2)
    elif case.get("quick"):
        quick[:2] = [True, True]
    if any(quick):
        limits = [ex_limit(T, *LIMITS[k], G) for T, k in zip(I.T, I.kinds)]
        limits[0] = limits[1] = limits[0] | limits[1]
    for n, T in enumerate(I.T):
        th = (ex_quicker(T, limits[n], fl, G, case.get("upwind", False)) if quick[n]
              else ex_mdfl(T, fl, G))
        if I.th is not None:
            th += I.th[n][:, 1:-1, 1:-1]
        out = torch.zeros(T.shape, dtype=F64, device=T.device)
        out[:, 1:-1, 1:-1] = ((fl.rho[:, 1:-1, 1:-1] * T[:, 1:-1, 1:-1].to(F64) + fl.dt * th)
                              * fl.rhor[:, 1:-1, 1:-1])
        del th
        outs.append(ex_vdiff(out, I.stf[n], I.btf[n], I.mix[1 if n == 1 else 0], None, fl, G))
        if case["kind"] == "plain" and G.cyclic:
            outs[-1][:, 1:-1, 0] = outs[-1][:, 1:-1, -2]
            outs[-1][:, 1:-1, -1] = outs[-1][:, 1:-1, 1]
    if case["kind"] == "plain":
        for L in limits:
            out = torch.zeros(I.T[0].shape, dtype=F64, device=I.T[0].device)
            out[:, :-1, :-1] = L.to(F64)
            outs.append(out)
    return outs


def halo(a, cyclic):
    if cyclic:
        a[..., 1:-1, 0] = a[..., 1:-1, -2]
        a[..., 1:-1, -1] = a[..., 1:-1, 1]
    return a


def ex_barotropic(I, nts, cgrid, press):
    """The time means and conv_rho_ud_t of nts subcycles (time stepping B)."""
    B, G = I.bt, I.G
    dt, r0 = G.dtbt, 1.0 / RHO0
    tm, um = G.tmask1, G.umask1
    dxr, dyr = 1.0 / (G.dxte + EPS40), 1.0 / (G.dytn + EPS40)

    def div(u):
        out = torch.zeros_like(tm)
        if cgrid:
            x, y = u[0] * G.dat * dxr, u[1] * G.dat * dyr
            out[1:, 1:] = (x[1:, 1:] - x[1:, :-1]) + (y[1:, 1:] - y[:-1, 1:])
        else:
            x, y = u[0] * G.dyu, u[1] * G.dxu
            xb, yb = 0.5 * (x[1:] + x[:-1]), 0.5 * (y[:, 1:] + y[:, :-1])
            out[1:, 1:] = (xb[:, 1:] - xb[:, :-1]) + (yb[1:] - yb[:-1])
        return out * G.datr

    def grad(p):
        g = torch.zeros(2, *p.shape, dtype=F64, device=p.device)
        if cgrid:
            g[0, :-1, :-1] = (p[:-1, 1:] - p[:-1, :-1]) * (dxr * B.tmasken[0])[:-1, :-1]
            g[1, :-1, :-1] = (p[1:, :-1] - p[:-1, :-1]) * (dyr * B.tmasken[1])[:-1, :-1]
        else:
            a, b = 0.5 * (p[1:] + p[:-1]), 0.5 * (p[:, 1:] + p[:, :-1])
            g[0, :-1, :-1] = (a[:, 1:] - a[:, :-1]) * (G.dxur * um)[:-1, :-1]
            g[1, :-1, :-1] = (b[1:] - b[:-1]) * (G.dyur * um)[:-1, :-1]
        return g

    def coriolis(u):
        F = torch.zeros_like(u)
        f, c = G.f, (slice(1, -1), slice(1, -1))
        v = u[1]
        F[(0,) + c] = 0.25 * (f[c] * (v[1:-1, 1:-1] + v[1:-1, 2:])
                              + f[:-2, 1:-1] * (v[:-2, 1:-1] + v[:-2, 2:]))
        v = u[0]
        F[(1,) + c] = -0.25 * (f[c] * (v[1:-1, 1:-1] + v[2:, 1:-1])
                               + f[1:-1, :-2] * (v[1:-1, :-2] + v[2:, :-2]))
        return F

    s = B.pme + B.river + B.source - B.smooth
    sf = tm * (GRAV * s + B.dpatm_dt) if press else tm * s
    cp, cc = (dt * GAMMA, dt) if press else (dt * GAMMA * r0, dt * r0)
    x, u = B.x.clone(), B.ud.clone()
    sx, su = B.x.clone(), torch.zeros_like(u)
    c1 = 0.5 * dt * G.f
    c2 = 1.0 / (1.0 + c1 * c1)
    if cgrid:
        F1 = F2 = coriolis(u)
    for it in range(1, nts + 1):
        d = div(u)
        t = -GRAV * d if press else -d * tm
        xs = x + cp * (t + sf)
        if not cgrid:
            halo(xs, G.cyclic)
        g = grad(tm * xs if press else B.rho_g * xs + B.patm)
        pf = -(r0 * B.thick * g) if press else -(B.thick * g)
        if cgrid:
            F0 = coriolis(u)
            acc = 23.0 / 12.0 * F0 - 16.0 / 12.0 * F1 + 5.0 / 12.0 * F2
            F1, F2 = F0, F1
            u = halo(u + dt * B.tmasken * (acc + pf + B.forcing), G.cyclic)
        else:
            t1 = u[0] + dt * (0.5 * G.f * u[1] + pf[0] + B.forcing[0])
            t2 = u[1] + dt * (-0.5 * G.f * u[0] + pf[1] + B.forcing[1])
            u = torch.stack([c2 * (t1 + c1 * t2), c2 * (t2 - c1 * t1)])
        d = div(u)
        t = -GRAV * d if press else -d * tm
        x = x + cc * (t + sf)
        sx += x
        su += (nts - it + 1) * u
    xb = halo(sx / (nts + 1.0), G.cyclic)
    ub = halo(su * (2.0 / (nts * (nts + 1.0))), G.cyclic)
    return [xb, ub, halo(-div(ub), G.cyclic)]


def ex_transports(I, case):
    G, B, press = I.G, I.bt, case["press"]
    z = torch.zeros_like(I.tend)
    a, b = I.u[0] * G.dyu * I.rho_dzu, I.u[1] * G.dxu * I.rho_dzu
    ue, vn = z.clone(), z.clone()
    ue[:, 1:] = 0.5 * (a[:, 1:] + a[:, :-1]) / G.dyte[1:]
    vn[..., 1:] = 0.5 * (b[..., 1:] + b[..., :-1]) / G.dxtn[:, 1:]
    dv = z.clone()
    x, y = G.dyte * ue, G.dxtn * vn
    dv[..., 1:] += x[..., 1:] - x[..., :-1]
    dv[:, 1:] += y[:, 1:] - y[:, :-1]
    dv *= G.datr * (levels(G) <= G.kmt)
    w = torch.zeros(G.nk + 1, *G.tmask1.shape, dtype=F64, device=z.device)
    w[0] = -(B.pme + B.river)
    for k in range(G.nk):
        w[k + 1] = (I.tend[k] + dv[k] + w[k]) * (G.kmt > k)
    um = (levels(G) <= G.kmu).to(F64)
    fb = (I.accel * um).sum(1) + G.umask1 * (I.smf - I.bmf)
    fb[:, 0], fb[:, -1] = 0.0, 0.0
    fb[..., 0], fb[..., -1] = (fb[..., -2], fb[..., 1]) if G.cyclic else (0.0, 0.0)
    s = I.conv + B.pme + B.river + B.source
    td = B.dpatm_dt + GRAV * G.tmask1 * s if press else G.tmask1 / RHO0 * s
    xp = torch.zeros_like(td)
    xp[1:-1, 1:-1] = (B.x + 1800.0 * td)[1:-1, 1:-1]
    halo(xp, G.cyclic)
    pb = xp + RHO0 * GRAV * G.ht if press else torch.zeros_like(td)
    src = RHO0 * GRAV * G.ht + I.anompb if press else B.x
    dte, dtw, dus, dun, daur = I.remap
    eu = torch.zeros_like(td)
    c, e, n, ne = ((slice(0, -1), slice(0, -1)), (slice(0, -1), slice(1, None)),
                   (slice(1, None), slice(0, -1)), (slice(1, None), slice(1, None)))
    eu[c] = (src[c] * dte[c] * dus[c] + src[e] * dtw[e] * dus[c] + src[n] * dte[n] * dun[c]
             + src[ne] * dtw[ne] * dun[c]) * daur[c] * G.umask1[c]
    halo(eu, G.cyclic)
    ps = B.rho_g * B.x + B.patm

    def grad(p):
        g = torch.zeros(2, *p.shape, dtype=F64, device=p.device)
        g[(0,) + c] = (0.5 * (p[e] + p[ne]) - 0.5 * (p[c] + p[n])) * (G.dxur * G.umask1)[c]
        g[(1,) + c] = (0.5 * (p[n] + p[ne]) - 0.5 * (p[c] + p[e])) * (G.dyur * G.umask1)[c]
        return g

    ga = grad(I.anompb) if press else torch.zeros(2, *td.shape, dtype=F64, device=td.device)
    return [ue, vn, dv, w, xp, td, pb, eu, ps, fb, grad(ps), ga]


def exact(case, seed):
    I = inputs(case, seed)
    kind = case["kind"]
    if kind == "ensemble":
        outs = [], [], [], []
        for P in I:
            t = ex_tracers(P, dict(kind="step"))
            x, u, _ = ex_barotropic(P, P.nts, False, False)
            for to, ts in zip(outs, (t[:2], t[2:], [x], [u])):
                to.extend(a.flatten() for a in ts)
        return [torch.cat(o) if o else None for o in outs]
    if kind in ("tracers", "plain"):
        return ex_tracers(I, case)
    if kind == "step":
        return ex_tracers(I, case) + ex_barotropic(I, case["nts"], False, False)
    if kind == "barotropic":
        return ex_barotropic(I, case["nts"], case["cgrid"], case["press"])
    if kind == "transports":
        return ex_transports(I, case)
    return [ex_vdiff(T, I.stf[n], I.btf[n], I.mix[1 if n == 1 else 0],
                     None if I.k33 is None else I.k33[n], I.flow, I.G) for n, T in enumerate(I.T)]
