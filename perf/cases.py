"""The measured work of this framework, through its public entry points.

A case is a plain dict.  Its "kind" says which call sequence a pass makes:

  steps    a model that stands in HBM is advanced by a few RK2 steps of a
           given length (a driver that samples the transient at fixed
           times), then its surface and its observation points are read
  request  a forward-model request on a kept model: reset, the coseismic
           set-up, adaptive RK2 steps, the surface and the points (a
           parameter search, or a server that reuses its models)
  batch    several models of one grid advanced together by Batch.step
  setup    the coseismic set-up alone (a static deformation model)
  green    greenfunctioncowling on device buffers (the C entry for callers
           that hold their fields on the GPU)
  host     one predictor stage through the per-routine entries on host
           arrays, as the relinked Fortran driver makes it

Units are km, MPa and years.  exact() recomputes a case in 64 bits with
torch alone.
"""
import math

import numpy as np
import torch

from relax_amd import load, workloads
from relax_amd import elastic3d, green, viscoelastic3d
from relax_amd.model import Batch
from relax_amd.structure import viscoelasticstructure
from relax_amd._lib import TENSOR_LAYER

LAM = MU = 3.0e4
GAM = 8.33e-4
BETA = 0.2
ALPHA = (LAM + MU) / (LAM + 2 * MU)
POINTS = 4096  # observation points of a model


def listed():
    return [
        # the smallest grid in use (tests, quick looks): launch latency
        case("steps", 64, 64, 64, rheology="maxwell", patches=3, steps=8, dt=0.02, dx=1.0),
        # the most frequent request of a rheology search
        case("request", 128, 128, 64, rheology="powerlaw", patches=5, steps=10, dx=1.0),
        # afterslip on a rate-strengthening plane with a power-law mantle
        case("steps", 256, 256, 128, rheology="afterslip", patches=1, steps=10, dt=0.002, dx=1.0),
        # the headline workload, with the launch shapes tuned as its benchmark does
        case("steps", 512, 512, 256, rheology="powerlaw", patches=40, steps=4, dt=0.01, dx=0.5, tuned=True),
        # Burgers rheology with a weak zone on the grid of the tutorial decks
        case("steps", 256, 256, 256, rheology="burgers", patches=4, steps=4, dt=0.01, dx=0.5),
        # the largest: a deep cubic grid
        case("steps", 512, 512, 512, rheology="maxwell", patches=8, steps=2, dt=0.02, dx=0.5),
        # a search over rheologies as one batch; an odd number of members
        case("batch", 128, 128, 128, members=11, patches=4, steps=10, dx=1.0),
        # a static coseismic model of a segmented rupture
        case("setup", 512, 512, 256, sources="shear", patches=40, dx=0.5),
        # a finely discretised slip model (patches below the Nyquist size), its
        # whole state kept by the caller
        case("setup", 256, 256, 128, sources="okada", patches=129, dx=1.0, whole=True),
        # volcanic unrest: dikes and point sources (images above the surface)
        case("setup", 256, 256, 128, sources="volcano", patches=5, dx=0.75),
        # one elastic solve of a caller with device-resident fields
        case("green", 512, 512, 256, dx=0.5),
        # the relinked Fortran driver on the plain CPU configuration's grid
        case("host", 128, 128, 64, rheology="maxwell", dx=0.5),
    ]


def case(kind, n1, n2, n3, **more):
    c = dict(kind=kind, n1=n1, n2=n2, n3=n3, **more)
    c.setdefault("dx2", c["dx"])
    what = c.get("sources") or c.get("rheology") or ("%d models" % c["members"] if kind == "batch" else "device")
    c["name"] = "%s %dx%dx%d %s" % (kind, n1, n2, n3, what)
    return c


def draw(rng):
    kind = rng.choice(("steps", "steps", "steps", "request", "batch", "setup", "setup", "green", "host"))
    most = dict(steps=2 ** 26, request=2 ** 23, batch=2 ** 21, setup=2 ** 25, green=2 ** 26, host=2 ** 21)[kind]
    while True:
        n1, n2 = (2 ** rng.randint(6, 10) for _ in range(2))
        n3 = 2 ** rng.randint(5, 9)
        if 2 ** 16 <= n1 * n2 * n3 <= most and max(n1, n2) <= 8 * n3 and n3 <= 2 * min(n1, n2):
            break
    dx = round(rng.uniform(0.4, 1.2), 2)
    more = dict(dx=dx, dx2=round(dx * rng.choice((1.0, 1.0, 0.8, 1.3)), 3))
    if kind == "steps":
        more.update(rheology=rng.choice(("maxwell", "powerlaw", "powerlaw", "burgers", "afterslip")),
                    patches=rng.randint(1, 23), steps=rng.randint(3, 12), dt=0.005)
        if more["rheology"] == "afterslip":
            more.update(patches=1, dt=0.002, dx2=dx)
        more["steps"] = max(1, min(more["steps"], 2 ** 27 // (n1 * n2 * n3)))
    elif kind == "request":
        more.update(rheology=rng.choice(("maxwell", "powerlaw")), patches=rng.randint(1, 9), steps=rng.randint(3, 19))
    elif kind == "batch":
        more.update(members=rng.randint(2, 13), patches=rng.randint(1, 5), steps=rng.randint(3, 10))
    elif kind == "setup":
        more["sources"] = rng.choice(("shear", "shear", "okada", "volcano"))
        more["patches"] = rng.randint(3, 47)
        if more["sources"] == "okada":
            more["patches"] = max(3, min(129, 2 ** 29 // (n1 * n2 * n3)))
            more["whole"] = n1 * n2 * n3 <= 2 ** 23
        elif more["sources"] == "volcano":
            more["patches"] = rng.randint(1, 7)
    elif kind == "host":
        more["rheology"] = "maxwell"
    c = case(kind, n1, n2, n3, **more)
    del c["name"]
    return c


# ------------------------------------------------------------ descriptions --
def spacing(c):
    return c["dx"], c["dx2"], c["dx"]


def spec(c, seed, member=0):
    """The description that workloads.build takes, of the case's seeded model."""
    rng = np.random.default_rng([seed, member])
    dx = c["dx"]
    # the horizontal half width and the depth of the half grid
    half = 0.5 * min(c["n1"] * dx, c["n2"] * c["dx2"])
    deep = 0.5 * c["n3"] * dx
    lid = math.floor(0.45 * c["n3"] / 2) * dx
    rheology = c.get("rheology") or ("powerlaw" if c["kind"] == "batch" else "maxwell")
    s = dict(sx1=c["n1"], sx2=c["n2"], sx3=c["n3"], dx=spacing(c), linear=None, nonlinear=None, friction=None,
             planes=None, deck=[], interval=1e30, odt=1.0, skip=1, tscale=1.0)
    size = 6 * dx
    for _ in range(c.get("patches", 0)):
        rake = rng.choice((0.0, 90.0)) + rng.uniform(-30, 30)
        s["deck"].append((rng.uniform(0.2e-3, 3e-3), rng.uniform(-0.5, 0.5) * half, rng.uniform(-0.5, 0.5) * half,
                          rng.uniform(0, 0.3) * deep, size, size, rng.uniform(0, 360), rng.uniform(30, 90), rake))
    if c.get("sources") == "okada":
        s["deck"] = [p[:4] + (dx, dx) + p[6:] for p in s["deck"]]
    if c.get("sources") == "volcano":
        s["tensile"] = [p[:6] + p[6:8] for p in s["deck"]]
        s["mogi"] = [(rng.uniform(1e-4, 1e-2), p[1], p[2], 4 * dx + p[3]) for p in s["deck"]]
        s["deck"] = []
    if rheology == "maxwell":
        s["linear"] = [(lid, workloads.gdot0(10 ** rng.uniform(18.5, 19.5)), 1.0, 0.0, 0.6, 0.0)]
    elif rheology == "powerlaw":
        # n = 3 below the lid, the fluidity growing with depth
        g = workloads.gdot0(10 ** rng.uniform(18.5, 19.5), 3.0)
        s["nonlinear"] = [(lid + dx * k, g * math.exp(dx * k / 10.0), 3.0, 0.0, 0.6, 0.0) for k in range(9)]
    elif rheology == "burgers":
        g = workloads.gdot0(10 ** rng.uniform(18.5, 19.5))
        s["linear"] = [(lid, g, 1.0, 0.0, 0.6, 0.0)]
        s["ltransient"] = [(lid, 20 * g, 1.0, 0.0, 0.6, 0.4 * MU)]
        # a vertical box of higher fluidity; its faces lie between grid points
        s["weak_linear"] = [(5 * g, -8.4 * dx, 0.3 * dx, lid - 3.4 * dx, 16.6 * dx, 9.2 * dx, 12.8 * c["dx2"], 0.0,
                             90.0)]
    else:
        # a creeping plane down dip of a thrust rupture
        s["nonlinear"] = [(lid, workloads.gdot0(1e18, 3.5), 3.5, 0.0, 0.6, 0.0)]
        dip, width = 20.0, round(0.125 * c["n3"]) * dx
        long = 2 * round(0.15 * half / dx) * dx
        down = width * math.sin(math.radians(dip)), width * math.cos(math.radians(dip))
        s["deck"] = [(rng.uniform(3e-5, 1.2e-4) * width, -0.25 * half, 0.0, 0.0, 0.5 * half, width, 0.0, dip, 90.0)]
        s["planes"] = [dict(x=-long / 2, y=-down[1], z=down[0], length=long, width=width, strike=0.0, dip=dip,
                            rake=-90.0)]
        s["friction"] = [(0.0, 1e-3, 1.0, 0.0, 0.6, 0.0)]
    # observation points on grid points of the top half
    i = np.stack([rng.integers(0, n, POINTS) for n in (c["n1"], c["n2"], c["n3"] // 2)], 1)
    return s, i


def coordinates(c, index):
    dx = np.array(spacing(c))
    n = np.array([c["n1"], c["n2"], c["n3"]])
    return np.where((index < n // 2) | (np.arange(3) == 2), index, index - n) * dx


def fields(c, seed, count, depth, device):
    """Smooth fields of a few bumps each, (count, depth, n2, n1)."""
    rng = np.random.default_rng(seed)
    out = torch.zeros((count, depth, c["n2"], c["n1"]), device=device)
    for a in out:
        for _ in range(3):
            g = [torch.as_tensor(np.exp(-0.5 * ((np.arange(n) - rng.uniform(0.2, 0.8) * n) / (0.04 * n + 2)) ** 2),
                                 dtype=torch.float32, device=device) for n in (depth, c["n2"], c["n1"])]
            a += float(rng.normal()) * g[0][:, None, None] * g[1][:, None] * g[2]
    return out


# ----------------------------------------------------------------- a pass --
def prepare(c, seed):
    kind = c["kind"]
    if kind == "green":
        h3 = c["n3"] // 2
        state = dict(c=c, f=torch.zeros((3, c["n3"], c["n2"], c["n1"] + 2), device="cuda"),
                     t=torch.zeros((3, c["n2"], c["n1"] + 2), device="cuda"))
        state["f"][:, :h3, :, :c["n1"]] = fields(c, seed, 3, h3, "cuda")
        state["t"][:, :, :c["n1"]] = fields(c, seed + 1, 3, 1, "cuda")[:, 0]
        state["w"] = torch.empty_like(state["f"])
        state["wt"] = torch.empty_like(state["t"])
        load().relax_hip_init(torch.cuda.current_device())
        return state
    if kind == "host":
        h3 = c["n3"] // 2
        s, _ = spec(c, seed)
        pad = (0, 2)
        return dict(c=c, structure=viscoelasticstructure(s["linear"], h3, c["dx"]),
                    prestress=np.zeros(h3, TENSOR_LAYER),
                    sig=np.ascontiguousarray(fields(c, seed, 6, h3, "cuda").movedim(0, -1).cpu().numpy()),
                    u=(1e-5 * torch.nn.functional.pad(fields(c, seed + 1, 3, h3, "cuda"), pad)).cpu().numpy())
    states = []
    for k in range(c.get("members", 1)):
        s, index = spec(c, seed, k)
        m = workloads.build(s)
        if c.get("tuned"):
            m.autotune()
        states.append(dict(m=m, spec=s, xyz=coordinates(c, index),
                           u=[np.zeros((c["n2"], c["n1"]), np.float32) for _ in range(3)]))
    state = dict(c=c, models=states)
    if kind == "batch":
        state["batch"] = Batch([s["m"] for s in states])
    return state


def observe(s, whole=False):
    """What a driver reads of a model at an output time: the surface and the
    observation points, or the whole state."""
    m = s["m"]
    if whole:
        state = m.download()
        return {k: state[k] for k in ("u1", "u2", "u3", "tau", "sig", "gamma")}
    m.surface(*s["u"])
    u, sig = m.points(s["xyz"])
    out = dict(surface=[a.copy() for a in s["u"]], u=u.astype(np.float32), sig=sig)
    if s["spec"]["planes"]:
        out["slip"] = m.get_patches()["slip"].astype(np.float32)
    return out


def run(state):
    c = state["c"]
    kind = c["kind"]
    if kind == "green":
        state["w"].copy_(state["f"])
        state["wt"].copy_(state["t"])
        rc = load().relax_greenfunctioncowling_noalloc(
            *[a.data_ptr() for a in state["w"]], *[a.data_ptr() for a in state["wt"]], c["n1"], c["n2"], c["n3"],
            *spacing(c), LAM, MU, GAM, torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError("greenfunctioncowling: status %d" % rc)
        return state["w"][:, :, :, :c["n1"]]
    if kind == "host":
        h3, dx = c["n3"] // 2, spacing(c)
        sig = state["sig"]
        moment = np.zeros_like(sig)
        tm = viscoelastic3d.viscouseigenstress(MU, state["structure"], state["prestress"], sig, moment, 1e7)
        f = np.zeros((3, c["n3"], c["n2"], c["n1"] + 2), np.float32)
        t = np.zeros((3, c["n2"], c["n1"] + 2), np.float32)
        elastic3d.equivalentbodyforce(moment, *dx, *[a[:h3] for a in f], *t)
        green.greenfunctioncowling(*f, *t, *dx, LAM, MU, GAM)
        half = tm / 20
        new = np.zeros_like(sig)
        elastic3d.tensorfieldadd(new, moment, 0.0, -half)
        v = state["u"].copy()
        for a, g in zip(v, f):
            elastic3d.fieldadd(a, np.ascontiguousarray(g[:h3]), None, half)
        elastic3d.stressupdate(*v, LAM, MU, *dx, new)
        return dict(moment=moment, v=v[:, :, :, :c["n1"]], sig=new)
    if kind == "batch":
        for _ in range(c["steps"]):
            state["batch"].step(info=False)
        return [observe(s) for s in state["models"]]
    s = state["models"][0]
    m = s["m"]
    if kind == "steps":
        m.run(c["steps"], dt_replay=[c["dt"]] * c["steps"])
    else:
        m.reset()
        workloads.configure(m, s["spec"])
        if kind == "request":
            m.run(c["steps"])
    return observe(s, c.get("whole"))


def work(c):
    """Bytes: a step reads and writes its state once per stage (displacement,
    stress, tau; gamma in the second), a solve its body force and its
    displacement.  Operations: the transforms and the pointwise laws."""
    n = c["n1"] * c["n2"] * c["n3"]
    h = n // 2
    solve = 6 * 2.5 * n * math.log2(n) + 100.0 * n
    steps = c.get("steps", 0) * c.get("members", 1)
    w = dict(bytes=272.0 * h * steps, flops=steps * (2 * solve + 400.0 * h))
    if c["kind"] == "green":
        w = dict(bytes=24.0 * n, flops=solve)
    elif c["kind"] == "host":
        # sig, u in; moment, v, sig out
        w = dict(bytes=4.0 * h * (6 + 3 + 6 + 3 + 6), flops=solve + 300.0 * h)
    elif c["kind"] in ("setup", "request"):
        pairs = 4000.0 * h * c["patches"] if c.get("sources") == "okada" else 300.0 * 1e3 * c["patches"]
        w["bytes"] += 4.0 * h * 15
        w["flops"] += solve + pairs
    return w


# ------------------------------------------------------- the same in 64 bits --
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def grid(c, depth):
    x = [torch.arange(n, device=DEV, dtype=torch.float64) for n in (c["n1"], c["n2"], depth)]
    x1, x2 = (torch.where(v < n / 2, v, v - n) * d for v, n, d in zip(x, (c["n1"], c["n2"]), spacing(c)))
    return x1, x2[:, None], x[2][:, None, None]


def solve64(c, f, t):
    """Elastic half-space response of a body force (3, depth, n2, n1) and a
    surface traction (3, n2, n1): the Fourier-domain solution with the
    correction of the surface traction and of buoyancy."""
    n1, n2, n3 = c["n1"], c["n2"], c["n3"]
    d1, d2, d3 = spacing(c)
    a, pi2 = ALPHA, 2 * math.pi

    def freq(n, d, half=False):
        i = torch.arange(n // 2 + 1 if half else n, device=DEV, dtype=torch.float64)
        return (i if half else torch.where(i < n / 2, i, i - n)) / (n * d)

    k1, k2, k3 = freq(n1, d1, True), freq(n2, d2)[:, None], freq(n3, d3)[:, None, None]
    U = torch.stack([torch.fft.fft(torch.fft.rfft2(x), n=n3, dim=0) for x in f]) * (d1 * d2 * d3)
    P = torch.fft.rfft2(t) * (d1 * d2)
    r2 = k1 * k1 + k2 * k2 + k3 * k3
    r2[0, 0, 0] = 1.0
    den = a / (MU * pi2 * pi2) / (r2 * r2)
    den[0, 0, 0] = 0.0
    kc = k1 * U[0] + k2 * U[1] + k3 * U[2]
    s = r2 * (1 + MU / (LAM + MU))
    for x, k in zip(U, (k1, k2, k3)):
        x.mul_(s).sub_(k * kc).mul_(den)
    del s, den, kc, r2
    q = 1j * pi2
    P[0] -= (q * MU * (k3 * U[0] + k1 * U[2])).sum(0) / (n3 * d3)
    P[1] -= (q * MU * (k3 * U[1] + k2 * U[2])).sum(0) / (n3 * d3)
    P[2] -= (q * ((LAM + 2 * MU) * k3 * U[2] + LAM * (k1 * U[0] + k2 * U[1]))
             - 2 * MU * a * GAM * U[2]).sum(0) / (n3 * d3)
    b = pi2 * torch.sqrt(k1 * k1 + k2 * k2)
    b[0, 0] = 1.0
    P[:, 0, 0] = 0.0
    b3 = (b * P[2] - 1j * (1 - a) * pi2 * (k1 * P[0] + k2 * P[1])) / (2 * a * MU * b ** 4 * (1 + GAM / b))
    Q = P / (2 * MU * b ** 3)
    bk = k1 * Q[0] + k2 * Q[1]
    fi = 2 * b / ((pi2 * k3) ** 2 + b * b)
    fk = fi * fi * pi2 * k3
    for j, k in ((0, k1), (1, k2)):
        U[j] += fi * (1j * k * a * b * pi2 * (1 - 1 / a) * b3 - 2 * b * b * Q[j] + k * a * pi2 ** 2 * bk)
        U[j] += fk * (k * a * b * pi2 * b3 - 1j * k * a * pi2 ** 2 * bk)
    U[2] += fi * (-b * b * b3) + fk * (1j * a * b * b * b3 + a * b * pi2 * bk)
    out = []
    for x in U:
        x = torch.fft.ifft(torch.fft.ifft(x, dim=0), dim=1) / (d1 * d2 * d3)
        x[..., 0].imag.zero_()
        x[..., -1].imag.zero_()
        out.append(torch.fft.irfft(x, n=n1))
    return torch.stack(out)


def diff(x, axis, d):
    """Centred differences: periodic along x1 (2) and x2 (1), one-sided at the
    top and the bottom along x3 (0)."""
    if axis:
        return (torch.roll(x, -1, axis) - torch.roll(x, 1, axis)) / (2 * d)
    y = torch.empty_like(x)
    y[1:-1] = (x[2:] - x[:-2]) / (2 * d)
    y[0], y[-1] = (x[1] - x[0]) / d, (x[-1] - x[-2]) / d
    return y


def hooke64(c, u):
    """C:eps(u), the six components 11, 12, 13, 22, 23, 33."""
    d = spacing(c)
    g = lambda i, j: diff(u[i], 2 - j, d[j])  # noqa: E731
    e = [g(0, 0), (g(1, 0) + g(0, 1)) / 2, (g(2, 0) + g(0, 2)) / 2, g(1, 1), (g(2, 1) + g(1, 2)) / 2, g(2, 2)]
    tr = LAM * (e[0] + e[3] + e[5])
    return torch.stack([2 * MU * x + (tr if i in (0, 3, 5) else 0) for i, x in enumerate(e)])


ROWS = ((0, 1, 2), (1, 3, 4), (2, 4, 5))


def force64(c, m):
    """-div(m) and m.e3 at the surface."""
    d = spacing(c)
    f = torch.stack([-sum(diff(m[r[j]], 2 - j, d[j]) for j in range(3)) for r in ROWS])
    return f, torch.stack([m[r[2]][0] for r in ROWS])


class Patch:
    """A rectangle of the deck (upper corner at the start of the strike,
    degrees) and the coordinates of the grid in its frame."""

    def __init__(self, c, line, x, turned=False):
        _, px, py, pz, self.W, self.L, strike, dip = line[:8]
        rake = line[8] if len(line) > 8 else 0.0
        if turned:
            rake = rake - 180.0 if rake >= 0 else rake + 180.0
        st, self.dip, rk = (math.radians(v) for v in (-90.0 - strike, 90.0 - dip, rake))
        cs, ss, cd, sd = math.cos(st), math.sin(st), math.cos(self.dip), math.sin(self.dip)
        self.cr, self.sr, self.cs, self.ss, self.cd, self.sd = math.cos(rk), math.sin(rk), cs, ss, cd, sd
        px += -self.W / 2 * ss + self.L / 2 * sd * cs
        py += -self.W / 2 * cs - self.L / 2 * sd * ss
        pz += self.L / 2 * cd
        self.x, self.y, self.z = px, py, pz
        self.Wp, self.Lp = (v * (1 + 2 * BETA) / 2 for v in (self.W, self.L))
        x1, x2, x3 = x
        xr = cs * px - ss * py
        self.xr, self.yr, self.zr = cd * xr - sd * pz, ss * px + cs * py, sd * xr + cd * pz
        xx = cs * x1 - ss * x2
        self.a, self.ai = cd * xx - sd * x3 - self.xr, cd * xx + sd * x3 - self.xr
        self.b = ss * x1 + cs * x2 - self.yr
        self.d, self.di = sd * xx + cd * x3 - self.zr, -sd * xx + cd * x3 + self.zr
        self.near = (self.a.abs() <= 7.01 * c["dx"]) | (self.ai.abs() <= 7.01 * c["dx"])
        self.n = (cd * cs, -cd * ss, -sd)
        self.r = (ss * self.cr + cs * sd * self.sr, cs * self.cr - ss * sd * self.sr, cd * self.sr)


def gauss(x, s):
    return torch.exp(-0.5 * (x / s) ** 2) / (math.sqrt(2 * math.pi) * s)


def gaussp(x, s):
    return -x / (s * s) * gauss(x, s)


def omega(x):
    y = ((1 - BETA) * x.abs() - 0.5 + BETA) / (2 * BETA)
    return torch.cos(math.pi * y.clamp(0, 0.5)) ** 2


def omegap(x):
    y = ((1 - BETA) * x.abs() - 0.5 + BETA) / (2 * BETA)
    return torch.where((y > 0) & (y < 0.5), -torch.sign(x) * math.pi * (1 - BETA) / (2 * BETA)
                       * torch.sin(2 * math.pi * y), torch.zeros_like(y))


def dyad(n, b):
    return [n[0] * b[0], (n[0] * b[1] + n[1] * b[0]) / 2, (n[0] * b[2] + n[2] * b[0]) / 2, n[1] * b[1],
            (n[1] * b[2] + n[2] * b[1]) / 2, n[2] * b[2]]


def aperture(p, h):
    return (gauss(p.a, h) * omega(p.d / p.L) + gauss(p.ai, h) * omega(p.di / p.L)) * omega(p.b / p.W)


def shear64(c, line, x, f, t, tau):
    """A tapered shear dislocation: its body force, its surface traction and
    its moment density."""
    p, h, s = Patch(c, line, x), c["dx"], -line[0]
    x1, x2, x3 = x
    box = ((x1 - p.x).abs() <= max(p.Wp, p.Lp)) & ((x2 - p.y).abs() <= max(p.Wp, p.Lp)) & p.near
    ap = aperture(p, h)
    for i, k in enumerate((2, 4, 5)):
        t[i] += torch.where(box[0], MU * s * dyad(p.n, p.r)[k] * ap[0], 0.0)
    here = box & (((x3 - p.z).abs() <= p.Lp) | ((x3 + p.z).abs() <= p.Lp))
    o2, o2p = omega(p.b / p.W), omegap(p.b / p.W)
    src = -MU * s * gaussp(p.a, h) * o2 * omega(p.d / p.L)
    dbl = -MU * s / p.W * gauss(p.a, h) * o2p * omega(p.d / p.L)
    dpc = -MU * s / p.L * gauss(p.a, h) * o2 * omegap(p.d / p.L)
    si = di = 0.0
    if math.radians(2.01) > p.dip:
        si = -MU * s * gaussp(p.ai, h) * o2 * omega(p.di / p.L)
        di = -MU * s / p.W * gauss(p.ai, h) * o2p * omega(p.di / p.L)
    cr, sr, cs, ss, cd, sd = p.cr, p.sr, p.cs, p.ss, p.cd, p.sd
    f[0] += torch.where(here, cr * ss * (src + si) + cr * cd * cs * (dbl + di) + sr * cs * (cd * dpc + sd * src), 0.0)
    f[1] += torch.where(here, cr * cs * (src + si) - cr * cd * ss * (dbl + di) - sr * ss * (cd * dpc + sd * src), 0.0)
    f[2] += torch.where(here, -cr * sd * (dbl - di) + sr * (cd * src - sd * dpc), 0.0)
    inside = ((x3 - p.z).abs() <= p.Lp) & ((x1 - p.x).abs() <= p.Wp) & ((x2 - p.y).abs() <= p.Wp) & p.near
    for a, e in zip(tau, dyad(p.n, p.r)):
        a += torch.where(inside, 2 * MU * s * e * ap, 0.0)


def tensile64(c, line, x, top, f, tau):
    """An opening crack with its image, over the full depth."""
    h, op = c["dx"], line[0]
    for full in (True, False):
        y = x if full else top
        p = Patch(c, line, y)
        x1, x2, x3 = y
        here = ((x1 - p.x).abs() <= p.Wp) & ((x2 - p.y).abs() <= p.Wp) & p.near
        if not full:
            ap = aperture(p, h)
            e = dyad([op * ap * v for v in p.n], [ap * v for v in p.n])
            tr = LAM * (e[0] + e[3] + e[5])
            here = here & ((x3 - p.z).abs() <= p.Lp)
            for k, a in enumerate(tau):
                a += torch.where(here, 2 * MU * e[k] + (tr if k in (0, 3, 5) else 0.0), 0.0)
            continue
        here = here & (((x3 - p.z).abs() <= p.Lp) | ((x3 + p.z).abs() <= p.Lp))
        o2, o2p = omega(p.b / p.W), omegap(p.b / p.W)
        part = []
        for a, d in ((p.a, p.d), (p.ai, p.di)):
            part.append((-op * (LAM + 2 * MU) * gaussp(a, h) * o2 * omega(d / p.L),
                         -op * LAM / p.W * gauss(a, h) * o2p * omega(d / p.L),
                         -op * LAM / p.L * gauss(a, h) * o2 * omegap(d / p.L)))
        (s, b, d), (si, bi, di) = part
        cs, ss, cd, sd = p.cs, p.ss, p.cd, p.sd
        f[0] += torch.where(here, cs * cd * (s + si) + ss * (b + bi) + cs * sd * (d + di), 0.0)
        f[1] += torch.where(here, -ss * cd * (s + si) + cs * (b + bi) - ss * sd * (d + di), 0.0)
        f[2] += torch.where(here, -sd * (s - si) + cd * (d - di), 0.0)


def mogi64(c, line, x, top, f, tau):
    """A point dilatation source with its image, over the full depth."""
    o, px, py, pz = line
    h = spacing(c)
    reach = 6 * max(h)
    x1, x2, x3 = x
    here = ((x1 - px).abs() <= reach) & ((x2 - py).abs() <= reach) & (((x3 - pz).abs() <= reach)
                                                                     | ((x3 + pz).abs() <= reach))
    k = -(LAM + 2 * MU / 3) * o
    g1, g2, z = gauss(x1 - px, h[0]), gauss(x2 - py, h[1]), gauss(x3 - pz, h[2]) + gauss(x3 + pz, h[2])
    f[0] += torch.where(here, k * gaussp(x1 - px, h[0]) * g2 * z, 0.0)
    f[1] += torch.where(here, k * g1 * gaussp(x2 - py, h[1]) * z, 0.0)
    f[2] += torch.where(here, k * g1 * g2 * (gaussp(x3 - pz, h[2]) - gaussp(x3 + pz, h[2])), 0.0)
    x1, x2, x3 = top
    here = ((x1 - px).abs() <= reach) & ((x2 - py).abs() <= reach) & ((x3 - pz).abs() <= reach)
    m = torch.where(here, -k * g1 * g2 * gauss(x3 - pz, h[2]), 0.0)
    for i in (0, 3, 5):
        tau[i] += m


class Model64:
    def __init__(self, c, s):
        self.c, self.s = c, s
        self.h3 = c["n3"] // 2
        x1, x2, x3 = grid(c, self.h3)
        self.x = (x1, x2, x3 * c["dx"])
        shape = (self.h3, c["n2"], c["n1"])
        new = lambda n, *sh: torch.zeros((n,) + sh, device=DEV, dtype=torch.float64)  # noqa: E731
        self.tau, t = new(6, *shape), new(3, *shape[1:])
        full = bool(s.get("tensile"))
        f = new(3, c["n3"] if full else self.h3, *shape[1:])
        for line in s["deck"]:
            shear64(c, line, self.x, f, t, self.tau)
        if full:
            x3 = grid(c, c["n3"])[2]
            y = (x1, x2, torch.where(x3 < self.h3, x3, x3 - c["n3"]) * c["dx"])
            for line in s["tensile"]:
                tensile64(c, line, y, self.x, f, self.tau)
            for line in s["mogi"]:
                mogi64(c, line, y, self.x, f, self.tau)
        self.u = solve64(c, f, t)[:, :self.h3].clone()
        self.sig = -self.tau + hooke64(c, self.u)
        self.E = new(6, *shape) if s.get("ltransient") else None
        self.plane = None
        if s["planes"]:
            p = s["planes"][0]
            line = (0.0, p["x"], p["y"], p["z"], p["length"], p["width"], p["strike"], p["dip"], p["rake"])
            self.plane = Patch(c, line, self.x, True)
            self.slip = torch.zeros((2,) + self.patch_index()[0].shape, device=DEV, dtype=torch.float64)
            self.rate = torch.zeros_like(self.slip)

    def patch_index(self):
        """Grid points nearest to the centres of the plane's patches."""
        p, c = self.plane, self.c
        down = lambda v: torch.ceil(v - 0.5).long()  # noqa: E731
        n2, n3 = math.ceil(p.W / c["dx2"] - 0.5), math.ceil(p.L / c["dx"] - 0.5)
        j = torch.arange(n2 * n3, device=DEV)
        y = p.yr + (j % n2 + 1 - n2 / 2 - 1).double() * c["dx2"]
        z = p.zr + (torch.div(j, n2, rounding_mode="floor") + 1 - n3 / 2 - 1).double() * c["dx"]
        x2p = p.cd * p.xr + p.sd * z
        X = (p.cs * x2p + p.ss * y, -p.ss * x2p + p.cs * y, -p.sd * p.xr + p.cd * z)
        return [down(v / d) for v, d in zip(X, spacing(c))]

    def table(self, key, col=1):
        v = torch.zeros(self.h3, device=DEV, dtype=torch.float64)
        for line in self.s[key]:
            v[int(round(line[0] / self.c["dx"])):] = line[col]
        return v[:, None, None]

    def friction(self, sig, m):
        """Rate-strengthening creep of the plane; returns the shortest time."""
        p, c, h = self.plane, self.c, self.c["dx"]
        x1, x2, x3 = self.x
        far = max(p.Wp, p.Lp)
        here = (((x3 - p.z).abs() <= p.Lp) | ((x3 + p.z).abs() <= p.Lp)) & p.near
        here = here & ((x1 - p.x).abs() <= far) & ((x2 - p.y).abs() <= far)
        t = [sum(sig[r[j]] * p.n[j] for j in range(3)) for r in ROWS]
        tn = sum(a * n for a, n in zip(t, p.n))
        ts = [a - tn * n for a, n in zip(t, p.n)]
        taus = torch.sqrt(sum(a * a for a in ts))
        tau = (taus + 0.6 * tn).clamp(min=0)
        here = here & (sum(a * r for a, r in zip(ts, p.r)) >= 0) & (taus > 0)
        rate = 2e-3 * torch.sinh((tau / 1.0).clamp(max=11.0))
        a = torch.where(here, 2 * MU * aperture(p, h) * rate, 0.0)
        for x, e in zip(m, dyad([v / torch.where(here, taus, 1.0) for v in ts], p.n)):
            x += a * e

    def creep(self, sig, dt):
        """Advance the patches' slip with the velocity at the stress sig; a
        patch that is pulled against its rake keeps its last velocity."""
        p = self.plane
        i1, i2, i3 = self.patch_index()
        c = self.c
        ok = (i3 >= 0) & (i3 < self.h3)
        s = sig[:, i3.clamp(0, self.h3 - 1), i2 % c["n2"], i1 % c["n1"]]
        t = [sum(s[r[j]] * p.n[j] for j in range(3)) for r in ROWS]
        tn = sum(a * n for a, n in zip(t, p.n))
        ts = [a - tn * n for a, n in zip(t, p.n)]
        taus = torch.sqrt(sum(a * a for a in ts))
        ok = ok & (sum(a * r for a, r in zip(ts, p.r)) >= 0) & (taus > 0)
        v = 2e-3 * torch.sinh((taus + 0.6 * tn).clamp(0, 11.0)) / torch.where(taus > 0, taus, 1.0)
        now = torch.stack([p.ss * ts[0] + p.cs * ts[1], -p.cs * p.sd * ts[0] + p.ss * p.sd * ts[1] - p.cd * ts[2]])
        self.rate = torch.where(ok, v * now, self.rate)
        self.slip += dt * self.rate

    def moment(self, sig, E):
        """The moment density rate, the transient strain rate and 1/(the
        largest strain rate factor)."""
        s, c = self.s, self.c
        dev = sig.clone()
        dev[[0, 3, 5]] -= (sig[0] + sig[3] + sig[5]) / 3
        norm = lambda d: torch.sqrt((d[0] ** 2 + d[3] ** 2 + d[5] ** 2) / 2 + d[1] ** 2 + d[2] ** 2 + d[4] ** 2)  # noqa
        m, Ed, tm = torch.zeros_like(sig), None, math.inf
        if s["linear"]:
            g = self.table("linear").expand(sig.shape[1:])
            if s.get("weak_linear"):
                dg, *line = s["weak_linear"][0]
                T = line.pop(5)
                p = Patch(c, [0.0] + line, self.x)
                g = g + dg * ((p.a.abs() <= T / 2) & (p.b.abs() <= p.W / 2) & (p.d.abs() <= p.L / 2))
            m += 2 * g * dev
            tm = 1 / float(torch.where(norm(dev) > 0, g, 0.0).max())
        if s["nonlinear"]:
            n = s["nonlinear"][0][2]
            g = self.table("nonlinear") * (norm(dev) / MU) ** (n - 1)
            m += 2 * g * dev
            tm = 1 / float(g.max())
        if E is not None:
            q = dev - 2 * self.table("ltransient", 5) * E
            g = self.table("ltransient")
            m += 2 * g * q
            Ed = g / MU * q
        if self.plane is not None:
            self.friction(sig, m)
        return m, Ed, tm

    def step(self, dt=None):
        c = self.c
        m, Ed, tm = self.moment(self.sig, self.E)
        dt = tm / 10 if dt is None else dt
        v = self.u + dt / 2 * solve64(c, *force64(c, m))[:, :self.h3]
        sig = -self.tau - dt / 2 * m + hooke64(c, v)
        m, Ed, _ = self.moment(sig, None if Ed is None else self.E + dt / 2 * Ed)
        if self.plane is not None:
            self.creep(sig, dt)
        self.u += dt * solve64(c, *force64(c, m))[:, :self.h3]
        self.tau += dt * m
        self.sig = -self.tau + hooke64(c, self.u)
        if Ed is not None:
            self.E += dt * Ed

    def observe(self, index):
        i1, i2, i3 = (torch.as_tensor(v, device=DEV) for v in index.T)
        out = dict(surface=[a[0].cpu().numpy() for a in self.u], u=self.u[:, i3, i2, i1].T.cpu().numpy(),
                   sig=self.sig[:, i3, i2, i1].T.cpu().numpy())
        if self.plane is not None:
            out["slip"] = torch.sqrt((self.slip ** 2).sum(0)).cpu().numpy()
        return out


def exact(c, seed):
    # Okada's closed form takes its arguments in single precision by its
    # interface (dc3d.f): it has no value in 64 bits
    if c.get("sources") == "okada":
        return None
    if c["kind"] == "green":
        h3 = c["n3"] // 2
        f = torch.zeros((3, c["n3"], c["n2"], c["n1"]), device=DEV, dtype=torch.float64)
        f[:, :h3] = fields(c, seed, 3, h3, DEV)
        return solve64(c, f, fields(c, seed + 1, 3, 1, DEV)[:, 0].double())
    if c["kind"] == "host":
        h3 = c["n3"] // 2
        s, _ = spec(c, seed)
        one = Model64(c, dict(s, deck=[]))
        sig = fields(c, seed, 6, h3, DEV).double()
        u = (1e-5 * fields(c, seed + 1, 3, h3, DEV)).double()
        m, _, tm = one.moment(sig, None)
        v = u + tm / 20 * solve64(c, *force64(c, m))[:, :h3]
        new = -tm / 20 * m + hooke64(c, v)
        return dict(moment=m.movedim(0, -1).contiguous(), v=v, sig=new.movedim(0, -1).contiguous())
    out = []
    for k in range(c.get("members", 1)):
        s, index = spec(c, seed, k)
        m = Model64(c, s)
        for _ in range(c.get("steps", 0)):
            m.step(c.get("dt"))
        out.append(m.observe(index))
    return out if c["kind"] == "batch" else out[0]
