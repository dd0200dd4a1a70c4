"""The work whose speed is measured: main-loop steps of single domains, batched
ensemble steps, windows on held wave products, and the learned wave
surrogate's inference and gradients, each through the package's public entry
points.

A case is a dict of plain values.  ``listed`` gives the named ones, ``draw``
one more of the same ranges, ``prepare`` what a program holds before the call
(a loaded domain, ensemble or network and its inputs, made from the seed
alone), ``run`` one pass, ``work`` the bytes and operations a pass cannot do
without, and ``exact`` the outputs of a first pass as plain torch gives them
in 64 bits.

Inputs: the barred rip-channel beach at mid-run, with wave energy spread
cos^2s about the mean direction and limited by the depth, currents, water
level, concentration and carried flow fields varying smoothly over some ten
cells, and wave-group records at the offshore boundary.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

PI = 3.14159265  # the model's constant
T0, TREP, NREC = 300.0, 9.0, 64  # time of boundary record 0, representative period, records

# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
STEP = dict(kind="step", loop="advance", nx=200, ny=50, nt=12, span=60.0, dx=5.0, morfac=1.0, zb_accum=0, wci=0.0,
            breakmodel=1, usesmago=1, Hm0=1.5, dir=0.0)


def _step(name, **kw):
    return dict(STEP, name=name, **kw)


def listed():
    return [
        # the small configuration (a profile-scale beach): the shortest calls,
        # run as the host driver runs its loop, running means included
        _step("driver loop 200x50x12", loop="driver"),
        # the same as one library call per iteration
        _step("step 200x50x12"),
        # the parameter defaults' half circle in 10-degree bins, an odd grid
        _step("step 413x287x18", nx=413, ny=287, nt=18, span=90.0, dx=4.0, Hm0=2.0, dir=-12.0),
        # wave-current interaction and the Baldock breaker, ragged sizes
        _step("step 777x389x24 currents", nx=777, ny=389, nt=24, dx=3.7, wci=1.0, breakmodel=2, usesmago=0, Hm0=2.5),
        # the morphology site: accelerated bed change, FP64 bed level
        _step("step 1024x512x24 morfac 10", nx=1024, ny=512, nt=24, dx=3.0, morfac=10.0, zb_accum=2, Hm0=3.0),
        # the large single domain of the benchmark
        _step("step 2048x1024x24", nx=2048, ny=1024, nt=24, dx=2.0, zb_accum=2, Hm0=3.0, dir=10.0),
        # storm-scenario ensembles: uneven domains, one training window of
        # steps with its window sums and sample
        dict(kind="ensemble", name="ensemble of 48", domains=48, nxmax=1024, nymax=512, steps=4),
        dict(kind="ensemble", name="ensemble of 12 small", domains=12, nxmax=256, nymax=160, steps=4),
        # the surrogate-assisted run between checkpoints: a window of steps
        # on held wave products
        dict(kind="window", name="products window 1024x512", nx=1024, ny=512, dx=3.0, seconds=1.0),
        # inference at the morphology site, from the fields to the products
        dict(kind="infer", name="infer 1x512x1024", n=1, H=512, W=1024),
        # training: the configuration's batch, and a short batch of a small grid
        dict(kind="train", name="train 64x256x256", n=64, H=256, W=256),
        dict(kind="train", name="train 3x48x256", n=3, H=48, W=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["ensemble", "window", "infer", "train"])
    if kind == "step":
        span = rng.choice([60.0, 60.0, 90.0])
        nt = rng.choice([12, 24, 24, 16, 9, 20] if span == 60.0 else [18, 18, 36, 12, 9])
        return dict(STEP, loop=rng.choice(["advance", "advance", "driver"]), nx=_log(rng, 64, 1900), ny=_log(rng, 37, 900),
                    nt=nt, span=span, dx=rng.choice([2.0, 3.0, 4.0, 5.0, round(rng.uniform(2.0, 5.0), 2)]),
                    morfac=rng.choice([1.0, 1.0, 10.0]), zb_accum=rng.choice([0, 0, 1, 2]),
                    wci=rng.choice([0.0, 0.0, 1.0]), breakmodel=rng.choice([1, 1, 2]), usesmago=rng.choice([1, 1, 0]),
                    Hm0=round(rng.uniform(0.5, 4.0), 2), dir=round(rng.uniform(-25.0, 25.0), 1))
    if kind == "ensemble":
        return dict(kind=kind, domains=_log(rng, 3, 48), nxmax=rng.randint(192, 1024), nymax=rng.randint(96, 512),
                    steps=rng.randint(1, 5))
    if kind == "window":
        return dict(kind=kind, nx=_log(rng, 256, 1300), ny=_log(rng, 128, 700), dx=rng.choice([2.0, 3.0, 4.0]),
                    seconds=round(rng.uniform(0.4, 1.2), 2))
    W = rng.choice([256, 256, 512, 1024])
    if kind == "infer":
        return dict(kind=kind, n=rng.randint(1, 4), H=16 * _log(rng, 1, 32), W=W)
    H = 16 * _log(rng, 1, 32)
    return dict(kind=kind, n=max(1, min(64, _log(rng, 1, 64), 64 * 65536 // (H * W))), H=H, W=W)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    return torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)


def _smooth(g, ny, nx, scale=10):
    """A random field of unit size varying over about ``scale`` cells."""
    a = torch.randn(1, 1, ny // scale + 2, nx // scale + 2, generator=g).to(_dev())
    return F.interpolate(a, size=(ny, nx), mode="bilinear", align_corners=True)[0, 0]


def _fields(c, seed):
    """Float32 fields of a domain at mid-run and its boundary records (double)."""
    g = _gen(seed)
    dev, nx, ny, dx = _dev(), c["nx"], c["ny"], c["dx"]
    x = torch.arange(nx, device=dev, dtype=torch.float64) * dx
    y = torch.arange(ny, device=dev, dtype=torch.float64) * dx
    xs = int(nx * 0.78) * dx
    crest = 1.0 + 0.5 * torch.sin(2 * math.pi * y / 200.0)
    elev = torch.clamp((x - xs) / 40.0, min=-20.0)[None, :] + crest[:, None] * torch.exp(-0.5 * ((x - (xs - 150.0)) / 20.0) ** 2)
    elev = elev + 0.05 * _smooth(g, ny, nx).double()
    zb = (-elev).float()
    wet = (zb > 0.05).float()
    zs = torch.maximum(torch.zeros_like(zb), -zb) + 0.05 * _smooth(g, ny, nx) * wet
    hh = torch.clamp(zb + zs, min=0.01)
    uu, vv = 0.3 * _smooth(g, ny, nx) * wet, 0.3 * _smooth(g, ny, nx) * wet
    f = dict(zb=zb, zs=zs, hh=hh, uu=uu, vv=vv, stdep=5.0 + _smooth(g, ny, nx),
             C=1e-3 * torch.rand(ny, nx, generator=g).to(dev) * wet)
    f["zsold"] = zs + 0.01 * _smooth(g, ny, nx) * wet
    f["uuold"], f["vvold"] = uu + 0.03 * _smooth(g, ny, nx) * wet, vv + 0.03 * _smooth(g, ny, nx) * wet
    f["qx"], f["qy"] = uu * hh, vv * hh
    f["vu"], f["uv"] = vv.clone(), uu.clone()
    f["ueu"], f["vev"] = uu - 0.02 * wet, vv.clone()
    f["vmageu"] = torch.sqrt(f["ueu"] ** 2 + f["vu"] ** 2)
    f["vmagev"] = torch.sqrt(f["uv"] ** 2 + f["vev"] ** 2)
    f["dzsdt"], f["rolthick"] = 0.02 * _smooth(g, ny, nx) * wet, 0.05 * torch.rand(ny, nx, generator=g).to(dev) * wet
    nt = c.get("nt", 12)
    th, dth = _theta(c)
    th, dth = torch.tensor(th, device=dev), float(dth)
    # energy spread cos^20 about the mean direction, depth limited
    D = torch.clamp(torch.cos(0.5 * (th - math.radians(c.get("dir", 0.0)))), min=0.0) ** 20
    D = D / (D.sum() * dth)
    Hr = torch.minimum(torch.full_like(hh, c.get("Hm0", 2.0) / math.sqrt(2.0)), 0.45 * hh)
    E = 1025.0 * 9.81 * Hr.double() ** 2 / 8.0 * torch.exp(0.25 * _smooth(g, ny, nx).double()) * wet.double()
    if "nt" in c:
        f["ee"] = (E[None] * D[:, None, None]).float()
        f["rr"] = f["ee"] * (0.15 * torch.rand(ny, nx, generator=g).to(dev))[None]
    # wave-group records: modulated energy and its bound long-wave flux
    t = torch.arange(NREC, dtype=torch.float64)[:, None] * c.get("dtbc", 1.0)
    yc = torch.arange(ny, dtype=torch.float64)[None, :] * dx
    env = torch.zeros(NREC, ny, dtype=torch.float64)
    for _ in range(6):
        u = torch.rand(3, generator=g, dtype=torch.float64)
        env += torch.cos(2 * math.pi * (t / (40.0 + 80.0 * u[0]) + u[1]) - (2 * u[2] - 1) * 2 * math.pi * yc / (ny * dx))
    env = 1.0 + 0.5 * env / math.sqrt(6.0)
    Eb = 1025.0 * 9.81 * c.get("Hm0", 2.0) ** 2 / 16.0
    S = (Eb * torch.clamp(env, min=0.05))[:, None, :] * D.cpu()[None, :, None]
    Q = torch.zeros(NREC, 4, ny, dtype=torch.float64)
    Q[:, 0] = -0.02 * (env - 1.0) * math.sqrt(9.81 * 10.0)
    return {k: v.float().contiguous() for k, v in f.items()}, S.contiguous(), Q


def _theta(c):
    """Bin centres and width (radians) as the model forms them."""
    nt, lo = c.get("nt", 12), -c.get("span", 60.0) * PI / 180.0
    dth = 2.0 * c.get("span", 60.0) / nt * PI / 180.0
    return np.array([np.float32(i * dth + lo + 0.5 * dth) for i in range(nt)], np.float64), dth


def _params(c):
    from xbeach_gpu_amd import default_params

    span = c.get("span", 60.0)
    return default_params(nx=c["nx"], ny=c["ny"], dx=c["dx"], thetamin=-span, thetamax=span, dtheta=2.0 * span / c.get("nt", 12),
                          D50=0.00025, morfac=c.get("morfac", 1.0), sedtrans=1, morphology=1, sedstart=0.0, CFL=0.7,
                          endtime=1e9, zb_accum=c.get("zb_accum", 0), wci=c.get("wci", 0.0),
                          breakmodel=c.get("breakmodel", 1), usesmago=c.get("usesmago", 1))


class _View:
    """A device array of the library, for torch.as_tensor; the tensor keeps
    this object, and this object the domain whose memory it is."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": "<f4", "version": 2}


class _Fields:
    """Device tensors over a domain's fields, one per buffer the library hands out."""

    def __init__(self, d):
        self.d, self.seen = d, {}

    def __call__(self, *names):
        out = {}
        for n in names:
            p = self.d.device_ptr(n)
            if p not in self.seen:
                self.seen[p] = torch.as_tensor(_View(self.d, p, self.d.shape_of(n)), device="cuda")
            out[n] = self.seen[p]
        return out


def _domain(c, seed):
    from xbeach_gpu_amd import Domain

    f, S, Q = _fields(c, seed)
    d = Domain(_params(c))
    for k, v in f.items():
        d.set(k, v.cpu().numpy())
    d.init_state(TREP)
    d.set_bnd_series(S.numpy(), Q.numpy())
    return d


def _ensemble_cases(c):
    """The domains of an ensemble: uneven grids, bins and sea states."""
    r = np.random.default_rng([c["domains"], c["nxmax"], c["nymax"]])
    out = []
    for k in range(c["domains"]):
        out.append(dict(nx=int(r.integers(c["nxmax"] // 4, c["nxmax"] + 1)), ny=int(r.integers(c["nymax"] // 4, c["nymax"] + 1)),
                        dx=float(np.float32(r.uniform(2.0, 5.0))), nt=int(r.choice([12, 24])), span=60.0,
                        Hm0=float(r.uniform(0.5, 4.0)), dir=float(r.uniform(-30.0, 30.0)), dtbc=600.0))
    return out


SUR = [(32, 32, 9, 1), (32, 32, 9, 1), (32, 64, 9, 1), (64, 64, 9, 1), (64, 128, 9, 1), (128, 128, 9, 1),
       (128, 256, 9, 1), (256, 256, 9, 1), (256, 128, 1, 0), (256, 128, 9, 1), (128, 128, 9, 1), (128, 64, 1, 0),
       (128, 64, 9, 1), (64, 64, 9, 1), (64, 32, 1, 0), (64, 32, 9, 1), (32, 32, 9, 1), (32, 5, 1, 0)]


def _sur_inputs(c, seed):
    """Parameters (a network some way into its training), fields, targets and
    normalisation of the surrogate's cases."""
    g = _gen(seed)
    P = []
    for cin, cout, taps, relu in SUR:
        P.append((torch.randn(taps * cout * cin, generator=g) * math.sqrt((2.0 if relu else 1.0) / (taps * cin))).float())
        P.append((0.05 * torch.randn(cout, generator=g)).float())
    n, H, W = c["n"], c["H"], c["W"]
    fields = torch.stack([torch.stack([_smooth(g, H, W, 16) for _ in range(4)]) for _ in range(n)])  # n, 4, H, W
    sea = torch.randn(n, 3, generator=g).to(_dev())
    x = torch.zeros(n, H, W, 8, device=_dev())
    x[..., :4] = fields.permute(0, 2, 3, 1)
    x[..., 4:7] = sea[:, None, None, :]
    t = torch.stack([torch.tanh(fields[:, 0] * fields[:, 1]), fields[:, 1] ** 2 - 0.7, torch.tanh(fields[:, 2]),
                     0.5 * fields[:, 2] + 0.5 * sea[:, 0, None, None].expand(n, H, W), fields[:, 3]], -1)
    return torch.cat(P), fields.contiguous(), sea, x.to(torch.bfloat16), t.to(torch.bfloat16).contiguous()


NORM14 = np.array([0.1, 0.0, 0.05, -0.05, 0.0, 0.0, 0.0, 1.1, 1.2, 0.9, 1.0, 1.0, 1.0, 1.0], np.float32)
NORM10 = np.array([0.6, 8.0, 6.0, 3.0, 0.5, 0.3, 6.0, 5.0, 8.0, 3.0], np.float32)


def _products(c, seed):
    """Normalised wave products of a network on the window's domain."""
    g = _gen(seed + 77)
    y = torch.stack([_smooth(g, c["ny"], c["nx"]) for _ in range(5)], -1)
    return torch.clamp(y, -1.5, 1.5).contiguous()


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
class State:
    pass


def prepare(case, seed):
    s = State()
    s.c = case
    kind = case["kind"]
    if kind in ("step", "window"):
        s.d = _domain(case, seed)
        s.fields = _Fields(s.d)
        s.t, s.dt = T0 + 1.0, 0.1
        s.d.state_save()
        if kind == "window":
            s.y = _products(case, seed)
            torch.cuda.synchronize()
    elif kind == "ensemble":
        from xbeach_gpu_amd.ensemble import Ensemble, RunSetup

        cases = _ensemble_cases(case)
        s.domains = [_domain(c, seed * 1000 + k) for k, c in enumerate(cases)]
        s.ens = Ensemble(s.domains, [RunSetup(T0 + 1.0, 0.1, 1e9, T0, c["dtbc"], TREP) for c in cases])
        s.meta = np.array([[c["Hm0"], 10.0, math.radians(c["dir"])] for c in cases], np.float32)
        s.raw = torch.empty(s.ens.window_enable(), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    else:
        from xbeach_gpu_amd.surrogate import Surrogate

        P, s.f, s.sea, s.x, s.t5 = _sur_inputs(case, seed)
        s.sur = Surrogate(case["n"], case["H"], case["W"])
        s.sur.set_params(P.numpy())
        if kind == "infer":
            s.sea = s.sea.cpu().tolist()
            s.x = torch.empty_like(s.x)
            s.y = torch.empty(case["n"], case["H"], case["W"], 5, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    return s


STEP_OUT = ("zs", "uu", "vv", "hh", "zb", "C", "stdep", "H", "urms", "thetamean", "DR", "Fx", "Fy", "ee", "rr")


def run(s):
    c = s.c
    if c["kind"] == "step":
        if s.t > T0 + NREC - 3.0:
            _again(s)
        if c["loop"] == "advance":
            s.t, s.dt = s.d.advance_resident(T0, 1.0, TREP, s.t, s.dt)
        else:
            _driver_iteration(s)
        return dict(s.fields(*STEP_OUT), t=s.t, dt=s.dt)
    if c["kind"] == "window":
        if s.t > T0 + NREC - 5.0:
            _again(s)
        s.d.set_wave_products(s.y.data_ptr(), NORM10, 0.1)
        s.d.reset_means()
        s.t, s.dt, n = s.d.advance_window(0, T0, 1.0, TREP, s.t + c["seconds"], 1e9, True, s.t, s.dt)
        s.d.divide_means(n)
        return dict(s.fields("zs", "uu", "vv", "hh", "zb", "C", "uumean", "vvmean", "zsmean", "Hmean"), n=n, dt=s.dt)
    if c["kind"] == "ensemble":
        for _ in range(c["steps"]):
            s.ens.step(1)
            s.ens.window_add()
        s.ens.window_sample(c["steps"], s.meta, s.raw.data_ptr())
        return s.raw
    if c["kind"] == "infer":
        from xbeach_gpu_amd import lib
        import ctypes as C

        norm = NORM14.ctypes.data_as(C.POINTER(C.c_float))
        cells = c["H"] * c["W"]
        for k in range(c["n"]):
            p = [s.f[k, j].data_ptr() for j in range(4)]
            rc = lib().xbg_sur_pack_inputs(*p, cells, *s.sea[k], norm, s.x[k].data_ptr(), None)
            if rc:
                raise RuntimeError("pack_inputs: %d" % rc)
        s.sur.forward(s.x.data_ptr(), c["n"], s.y.data_ptr())
        return s.y
    loss = s.sur.backward(s.x.data_ptr(), s.t5.data_ptr(), c["n"])
    return dict(loss=loss, grads=s.sur.grads())


def _again(s):
    """At the end of the block of records (some hundred steps): its start again."""
    s.d.state_restore()
    s.t, s.dt = T0 + 1.0, 0.1


def _driver_iteration(s):
    """The host driver's loop body: limits, time step, boundary record, step, running means."""
    from xbeach_gpu_amd import next_dt

    dtf, dtw = s.d.cfl()
    s.dt = next_dt(dtf, dtw, 1, s.dt, s.t, 1e30, 1e30)
    s.t += s.dt
    rec = int(math.floor(s.t - T0))
    s.d.use_bnd_record(rec, s.t - (rec + T0), 1.0, TREP)
    s.d.step(s.dt, s.t)
    s.d.accumulate_means()


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _step_work(nx, ny, nt, zb_accum, wave=True):
    # carried state read and written once; per bin two fields advected in
    # three directions, dissipation and the moments, per cell the flow and
    # sediment stencils
    n = nx * ny
    return n * ((16 * nt if wave else 0) + 104 + (16 if zb_accum == 2 else 0)), n * ((130 * nt if wave else 0) + 700)


def work(case):
    k = case["kind"]
    if k == "step":
        b, f = _step_work(case["nx"], case["ny"], case["nt"], case["zb_accum"])
    elif k == "window":
        steps = case["seconds"] / (0.0248 * case["dx"])  # dt from the offshore depth of 20 m
        b, f = _step_work(case["nx"], case["ny"], 0, 0, wave=False)
        b, f = steps * b, steps * f
    elif k == "ensemble":
        # domains of the mean size and bin count of the range
        n = case["domains"] * (0.625 * case["nxmax"]) * (0.625 * case["nymax"])
        b, f = case["steps"] * n * (16 * 18 + 104 + 64) + n * 80, case["steps"] * n * (130 * 18 + 700)
    else:
        p = case["n"] * case["H"] * case["W"]
        level = [0, 0, 1, 1, 2, 2, 3, 3, 3, 2, 2, 2, 1, 1, 1, 0, 0, 0]
        macs = [p / 4 ** l * taps * cin * cout for (cin, cout, taps, _), l in zip(SUR, level)]
        macs[0] *= 8.0 / 32.0  # eight input channels
        act = sum(p / 4 ** l * cout * 2 for (_, cout, _, _), l in zip(SUR, level))
        b, f = p * 16 + p * 20, 2 * sum(macs)
        if k == "train":
            # every activation is written, and read again by the backward
            b, f = p * 26 + 2 * act, 3 * f - 2 * macs[0]
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
class _Model:
    """A domain in torch float64: the surf-beat step's equations on whole arrays."""

    def __init__(self, c, seed):
        f, S, Q = _fields(c, seed)
        self.c = c
        self.nx, self.ny, self.dx = c["nx"], c["ny"], float(np.float32(c["dx"]))
        self.dtbc, self.S, self.Q = c.get("dtbc", 1.0), S, Q
        dev = _dev()
        self.IX = torch.arange(self.nx, device=dev)
        self.IY = torch.arange(self.ny, device=dev)
        for k, v in f.items():
            setattr(self, k, v.double())
        self.zb = self.zb.clone()
        self.umean = torch.zeros(self.ny, dtype=torch.float64, device=dev)
        self.rho, self.g, self.eps, self.CFL = 1025.0, 9.81, 0.01, 0.7
        self.beta, self.gammax, self.hwci, self.wci = 0.15, 2.0, 0.1, c.get("wci", 0.0)
        self.nuh = 0.3 if c.get("usesmago", 1) == 1 else 1.0
        self.sig = 2 * PI / TREP
        self.dtwave = None
        self.depths()

    # values at the clamped neighbour (dx, dy)
    def at(self, a, dx, dy=0):
        if dx:
            a = a[..., (self.IX + dx).clamp(0, self.nx - 1)]
        if dy:
            a = a[..., (self.IY + dy).clamp(0, self.ny - 1), :]
        return a

    def rows(self, a):
        """Rows 0 and ny-1 from rows 1 and ny-2."""
        a = a.clone()
        a[..., 0, :], a[..., -1, :] = a[..., 1, :], a[..., -2, :]
        return a

    def depths(self):
        def face(vel, dx, dy):
            hb = torch.maximum(-self.zb, -self.at(self.zb, dx, dy))
            z, zn = self.zs, self.at(self.zs, dx, dy)
            h = torch.where(vel > 0, z - hb, torch.where(vel < 0, zn - hb, (torch.maximum(z, zn) - hb).clamp(min=self.eps)))
            return h.clamp(min=0.0)

        self.hu, self.hv = face(self.uu, 1, 0), face(self.vv, 0, 1)

    def next_dt(self, t, prev, stop=1e30, with_wave=True):
        dt = 0.5 * float((self.CFL * self.dx / torch.sqrt(9.81 * self.hh)).min())
        if with_wave and self.dtwave is not None:
            dt = min(dt, 0.5 * self.dtwave)
        diff = dt - prev
        if abs(diff) / prev > 0.1:
            dt = prev * (1 + math.copysign(0.1, diff))
        n = math.ceil((stop - t) / dt)
        return (stop - t) / n if n > 0 else dt

    def step(self, t, dt, wave=True):
        """One step that ends at time t."""
        rec = int(math.floor((t - T0) / self.dtbc))
        w = (t - (rec * self.dtbc + T0)) / self.dtbc
        lerp = lambda A: (A[rec] + w * (A[rec + 1] - A[rec])).to(_dev())  # noqa: E731
        St, q = lerp(self.S), lerp(self.Q)
        taper = min(t / 100.0, 1.0)
        if wave:
            self.dispersion()
        # offshore boundary
        fac = 0.25 / TREP * dt
        ui = q[0] * taper / self.zb[:, 0]
        ur = -torch.sqrt(self.g / self.hh[:, 0]) * self.zs[:, 1]
        self.umean = fac * self.uu[:, 0].mean() + self.umean * (1 - fac)
        self.uu, self.vv, self.zs = self.uu.clone(), self.vv.clone(), self.zs.clone()
        self.uu[:, 0] = 2 * ui + ur + self.umean
        self.zs[:, 0], self.vv[:, 0] = self.zs[:, 1], self.vv[:, 1]
        if wave:
            self.wave(St * taper, dt)
        self.flow(dt)
        self.sediment(dt)

    def dispersion(self):
        h, sig = self.hh, self.sig
        phi = (1 + math.sqrt(5.0)) / 2
        L0 = 2 * math.pi * self.g / sig ** 2
        L1 = torch.full_like(h, L0)
        act = torch.ones_like(h, dtype=torch.bool)
        for n in range(1, 200):
            L2 = L0 * torch.tanh(2 * PI * h / L1)
            err = (L2 - L1).abs()
            L1 = torch.where(act, L1 / (phi + 1) + L2 * (phi / (phi + 1)), L1)
            act = act & (err > 1e-4)
            if n % 4 == 0 and not bool(act.any()):
                break
        self.k = 2 * PI / L1
        self.cc = sig / self.k
        kh = (self.k * h).clamp(max=10.0)
        self.cg = self.cc * (0.5 + kh / torch.sinh(2 * kh))

    @staticmethod
    def up2(a, b):
        v = 1.5 * a - 0.5 * b
        return torch.where(v < 0, a, v)

    def advect(self, e, S, ct, cs, sn, dth):
        """x, y and theta upwind flux divergence of e[nt, ny, nx] at speed S."""
        at, nt = self.at, e.shape[0]
        wc = self.wci * (self.hh / self.hwci).clamp(max=1.0)
        out = torch.zeros_like(e)
        for i in range(nt):
            b = e[i]
            for c_, vel, ax in ((cs[i], self.uu, 0), (sn[i], self.vv, 1)):
                A = (lambda f, k: at(f, k)) if ax == 0 else (lambda f, k: at(f, 0, k))
                cp = 0.5 * (S * c_ + vel * wc + A(S, 1) * c_ + A(vel, 1) * wc)
                cm = 0.5 * (S * c_ + vel * wc + A(S, -1) * c_ + A(vel, -1) * wc)
                fp = self.up2(torch.where(cp > 0, b, A(b, 1)), torch.where(cp > 0, A(b, -1), A(b, 2))) * cp
                fm = self.up2(torch.where(cm > 0, A(b, -1), b), torch.where(cm > 0, A(b, -2), A(b, 1))) * cm
                out[i] += (fp - fm) / self.dx
        for i in range(nt - 1):
            cb = 0.5 * (ct[i] + ct[i + 1])
            fr = cb * self.up2(torch.where(cb > 0, e[i], e[i + 1]),
                               torch.where(cb > 0, e[max(i - 1, 0)], e[min(i + 2, nt - 1)]))
            out[i] += fr / dth
            out[i + 1] -= fr / dth
        return out

    def wave(self, St, dt):
        c, at, g, rho = self.c, self.at, self.g, self.rho
        th, dth = _theta(c)
        cs, sn, nt = np.cos(th), np.sin(th), len(th)
        h, k, cc, cg, sig = self.hh, self.k, self.cc, self.cg, self.sig
        e = self.ee.clone()
        e[:, :, 0] = St
        e = e.clamp(min=0.0) / sig
        r = self.rr
        ddx = ((self.IX + 1).clamp(max=self.nx - 1) - (self.IX - 1).clamp(min=0)).double() * self.dx
        ddy = (((self.IY + 1).clamp(max=self.ny - 1) - (self.IY - 1).clamp(min=0)).double() * self.dx)[:, None]
        sx = lambda f: (at(f, 1) - at(f, -1)) / ddx  # noqa: E731
        sy = lambda f: (at(f, 0, 1) - at(f, 0, -1)) / ddy  # noqa: E731
        hx, hy, ux, uy, vx, vy = sx(h), sy(h), sx(self.uu), sy(self.uu), sx(self.vv), sy(self.vv)
        sk = sig / torch.sinh(2 * (k * h).clamp(max=10.0))
        w = self.wci * (h / self.hwci).clamp(max=1.0)
        ct = torch.stack([(sk * (hx * sn[i] - hy * cs[i]) + w * (cs[i] * (sn[i] * ux - cs[i] * uy) + sn[i] * (sn[i] * vx - cs[i] * vy))
                           ).clamp(-0.25 * sig, 0.25 * sig) for i in range(nt)])
        self.dtwave = min(9999999.9, float(self.CFL * dth / ct.abs().max()))
        e = e - dt * self.advect(e, cg, ct, cs, sn, dth)
        r = r - dt * self.advect(r, cc, ct, cs, sn, dth)
        wet = (h > self.eps)
        edge = torch.ones_like(h)
        edge[0], edge[-1] = wet[0].double(), wet[-1].double()
        e, r = self.rows(e) * edge, self.rows(r) * edge
        e = (e * sig).clamp(min=0.0)
        Ht = torch.sqrt(e.sum(0) * dth / (rho * g / 8))
        e = e / ((Ht / (self.gammax * h)) ** 2).clamp(min=1.0)
        Ht = torch.minimum(Ht, self.gammax * h)
        E = rho * g * Ht ** 2 / 8
        if c.get("breakmodel", 1) == 1:
            Hr = torch.sqrt(E * 8 / rho / g)
            Qb = (1 - torch.exp((-(Hr / 0.6 / h) ** 8).clamp(min=-100.0))).clamp(max=1.0)
            D = Qb * 2 / TREP * E * Hr / h
        else:
            Hr = Ht
            Hb = 0.88 / k * torch.tanh(0.6 * k * h / 0.88)
            D = 0.25 * torch.exp(-(Hb / Ht.clamp(min=1e-5)) ** 2) * rho / TREP * g * (Hb ** 2 + Ht ** 2)
        uorb = PI * Hr / (TREP * torch.sinh((k * h).clamp(max=10.0)))
        D = D + 0.66666666 / PI * rho * 0.001 * uorb ** 3
        self.Dw = D
        R, DR = torch.zeros_like(h), torch.zeros_like(h)
        for i in range(nt):
            cx, cy = cc * cs[i] + self.uu * w, cc * sn[i] + self.vv * w
            dd = e[i] * D / E.clamp(min=1e-7)
            rd = 2 * g * self.beta * r[i] / torch.sqrt(cx ** 2 + cy ** 2)
            e[i] = torch.where(wet, (e[i] - dt * dd).clamp(min=0.0), 0.0)
            r[i] = torch.where(wet, (r[i] + dt * (dd - rd)).clamp(min=0.0), 0.0)
            DR = torch.where(wet, DR + rd, 0.0)
            R = R + r[i]
        self.R, self.DR = R * dth, DR * dth
        e = self.rows(e) * edge
        self.ee, self.rr = e, r
        m = lambda f, v: torch.einsum("i,iyx->yx", torch.tensor(f, device=h.device), v)  # noqa: E731
        nn, sume = cg / cc, e.sum(0)
        Sxx = (nn * m(1 + cs * cs, e) - 0.5 * sume) * dth + m(cs * cs, r) * dth
        Syy = (nn * m(1 + sn * sn, e) - 0.5 * sume) * dth + m(sn * sn, r) * dth
        Sxy = nn * m(sn * cs, e) * dth + m(sn * cs, r) * dth
        sm = sume.clamp(min=1e-5)
        self.thetamean = m(th, e) / sm
        self.H = torch.sqrt(sm * dth / (rho * g / 8))
        self.urms, ust = self.drift(sm * dth)
        # forces and their boundary rules
        Fx = -(at(Sxx, 1) - Sxx) / self.dx - 0.5 * (at(Sxy, 0, 1) + at(Sxy, 1, 1) - at(Sxy, 0, -1) - at(Sxy, 1, -1)) / (2 * self.dx)
        Fy = -(at(Syy, 0, 1) - Syy) / self.dx - 0.5 * (at(Sxy, 1) + at(Sxy, 1, 1) - at(Sxy, -1) - at(Sxy, -1, 1)) / (2 * self.dx)
        wd = wet.double()
        self.Fx = self.rows(Fx) * edge
        f0, u0 = Fy[:, 1] * wd[:, 0], ust[:, 1] * wd[:, 0]
        self.Fy, self.ust = self.rows(Fy) * edge, self.rows(ust) * edge
        self.Fy[:, 0], self.ust[:, 0] = f0, u0

    def drift(self, E):
        hi = self.hh.clamp(min=0.2)
        ci = self.cc.clamp(min=math.sqrt(0.2 * self.g))
        uorb = PI * self.H / TREP / torch.sinh((self.k.clamp(min=0.01) * hi).clamp(max=10.0))
        return uorb / math.sqrt(2.0), (E + 2 * self.R) / ci / self.rho / hi

    def products(self, y):
        """The wave fields from normalised H, Dw, DR, Fx, Fy [ny, nx, 5]."""
        self.dispersion()
        v = self.rows((y.double() * torch.tensor(NORM10[5:], device=y.device).double()
                       + torch.tensor(NORM10[:5], device=y.device).double()).permute(2, 0, 1))
        wet = (self.hh > self.eps).double()
        Hp, Hm = v[0].clamp(min=0.0), self.gammax * self.hh
        sc = torch.where(Hp > Hm, (Hm / Hp) ** 2, 1.0) * wet
        self.H = torch.minimum(Hp, Hm) * wet
        self.DR, self.Fx, self.Fy = v[2].clamp(min=0.0) * sc, v[3] * sc, v[4] * sc
        self.R = self.DR * self.cc / (2 * self.g * self.beta)
        self.urms, ust = self.drift(self.rho * self.g * self.H ** 2 / 8)
        self.ust, self.thetamean = ust * wet, torch.full_like(self.hh, 0.1)

    def flow(self, dt):
        at, dx, g, rho, eps = self.at, self.dx, self.g, self.rho, self.eps
        h, u, v, zs, zb, hu, hv = self.hh, self.uu, self.vv, self.zs, self.zb, self.hu, self.hv
        hum = (0.5 * (h + at(h, 1))).clamp(min=eps)
        hvm = (0.5 * (h + at(h, 0, 1))).clamp(min=eps)
        wu = ((hu > eps) & (0.5 * (h + at(h, 1)) > eps)).double()
        wv = ((hv > eps) & (0.5 * (h + at(h, 0, 1)) > eps)).double()
        nuh = h * (self.DR / rho) ** (1 / 3)
        if self.c.get("usesmago", 1) == 1:
            a = (u - at(u, -1)) / dx
            b = 0.5 * (at(u, 0, 1) - at(u, 0, -1) + at(u, -1, 1) - at(u, -1, -1)) / dx
            d = (v - at(v, 0, -1)) / dx
            e = 0.5 * (at(v, 1) - at(v, -1) + at(v, 1, -1) - at(v, -1, -1)) / dx
            nuh = torch.maximum(self.nuh ** 2 * dx ** 2 * torch.sqrt(2 * a * a + 2 * d * d + (b + e) ** 2), nuh)
        else:
            nuh = nuh.clamp(min=self.nuh)
        pos = lambda q, val: torch.where(q > 0, val, 0.0)  # noqa: E731
        cf = 0.01
        # u momentum
        ul, ur, ub, ut = at(u, -1), at(u, 1), at(u, 0, -1), at(u, 0, 1)
        q = 0.5 * (hu * u + at(hu, -1) * ul)
        adv = pos(q, torch.where(u - ul > 0.5, 0.5 * (ul + u) * (u - ul) / dx, q / hum * (u - ul) / dx))
        q = -0.5 * (hu * u + at(hu, 1) * ur)
        adv = adv + pos(q, torch.where(ur - u > 0.5, -0.5 * (ur + u) * (u - ur) / dx, q / hum * (u - ur) / dx))
        vb, vbr, vr = at(v, 0, -1), at(v, 1, -1), at(v, 1)
        q = 0.5 * (vb * at(hv, 0, -1) + vbr * at(hv, 1, -1))
        adv = adv + pos(q, torch.where(v - vb > 0.5, 0.5 * (vb + vbr) * (u - ub) / dx, q / hum * (u - ub) / dx))
        q = -0.5 * (v * hv + vr * at(hv, 1))
        adv = adv + pos(q, torch.where(at(v, 0, 1) - v > 0.5, -0.5 * (v + vr) * (u - ut) / dx, q / hum * (u - ut) / dx))
        vis = (at(nuh, 1) * at(h, 1) * (ur - u) / dx - nuh * h * (u - ul) / dx) / dx / hum
        n1 = 0.25 * (nuh + at(nuh, 1) + at(nuh, 1, 1) + at(nuh, 0, 1))
        n2 = 0.25 * (nuh + at(nuh, 1) + at(nuh, 1, -1) + at(nuh, 0, -1))
        d1 = n1 * 0.5 * (hvm + at(hvm, 1)) * (ut - u) / dx
        hb = at(h, 0, -1)
        ym = (self.IY - 1).clamp(min=0)
        hbt = h[(ym + 1).clamp(max=self.ny - 1)]
        g2 = (0.5 * (hb + hbt)).clamp(min=eps)
        d2 = n2 * 0.5 * (g2 + at(g2, 1)) * (u - ub) / dx
        vis = vis + (d1 - d2) / dx / hum * at(wu, 0, 1) * at(wu, 0, -1)
        tau = cf * rho * self.ueu * torch.sqrt(1.3456 * self.urms ** 2 + self.vmageu ** 2)
        un = u - dt * (adv - vis + g * (at(zs, 1) - zs) / dx + tau / (rho * hu) - self.Fx / (rho * hum.clamp(min=0.2)))
        un = torch.where(wu > 0, un, 0.0)
        un[:, 0] = u[:, 0]
        un = self.rows(un)
        # v momentum, on the new u
        vl, vt = at(v, -1), at(v, 0, 1)
        unl, untl, unt = at(un, -1), at(un, -1, 1), at(un, 0, 1)
        q = 0.5 * (unl * at(hu, -1) + untl * at(hu, -1, 1))
        adv = pos(q, torch.where(un - unl > 0.5, 0.5 * (unl + untl) * (v - vl) / dx, q / hvm * (v - vl) / dx))
        q = -0.5 * (un * hu + unt * at(hu, 0, 1))
        unr = at(un, 1)
        adv = adv + pos(q, torch.where(unr - un > 0.5, -0.5 * (un + unr) * (v - vr) / dx, q / hvm * (v - vr) / dx))
        q = 0.5 * (v * hv + vb * at(hv, 0, -1))
        adv = adv + pos(q, torch.where(v - vb > 0.5, 0.5 * (vb - v) * (v - vb) / dx, q / hvm * (v - vb) / dx))
        q = -0.5 * (hv * v + at(hv, 0, 1) * vt)
        adv = adv + pos(q, torch.where(vt - v > 0.5, -0.5 * (vt + v) * (v - vt) / dx, q / hvm * (v - vt) / dx))
        vis = (at(nuh, 0, 1) * at(h, 0, 1) * (vt - v) / dx - nuh * h * (v - vb) / dx) / dx / hvm * at(wv, 0, 1) * at(wv, 0, -1)
        n2 = 0.25 * (nuh + at(nuh, -1) + at(nuh, -1, 1) + at(nuh, 0, 1))
        d1 = n1 * 0.5 * (hum + at(hum, 0, 1)) * (vr - v) / dx
        d2 = n2 * 0.5 * (at(hum, -1) + at(hum, -1, 1)) * (v - vl) / dx
        vis = vis + (d1 - d2) / dx / hvm * at(wv, 1) * at(wv, -1)
        tau = cf * rho * self.vev * torch.sqrt(1.3456 * self.urms ** 2 + self.vmagev ** 2)
        vn = v - dt * (adv - vis + g * (at(zs, 0, 1) - zs) / dx + tau / (rho * hv) - self.Fy / (rho * hvm.clamp(min=0.2)))
        vn = torch.where(wv > 0, vn, 0.0)
        vn[:, 0], vn[-1], vn[-2] = v[:, 0], v[-1], v[-2]
        vn[0], vn[-2] = vn[1], vn[-3]
        self.correct(dt, un, vn, hum, hvm)
        self.depths()
        self.levels(dt)
        # Lagrangian and Eulerian velocities at the other face
        u, v, tm, us = self.uu, self.vv, self.thetamean, self.ust
        vu = 0.25 * (at(v, 0, -1) + v + at(v, 1, -1) + at(v, 1)) * wu
        uv = 0.25 * (at(u, -1) + u + at(u, -1, 1) + at(u, 0, 1)) * wv
        sx, cx = us * torch.sin(tm), us * torch.cos(tm)
        ue, ve = u - 0.5 * (cx + at(cx, 1)) * wu, vu - 0.5 * (sx + at(sx, 1)) * wu
        vev, uev = v - 0.5 * (sx + at(sx, 0, 1)) * wv, uv - 0.5 * (cx + at(cx, 0, 1)) * wv
        self.uuold, self.vvold, self.zsold = u, v, self.zs
        self.uv, self.vu, self.ueu, self.vev = (self.rows(a) for a in (uv, vu, ue, vev))
        self.vmageu = self.rows(torch.sqrt(ue ** 2 + ve ** 2))
        self.vmagev = self.rows(torch.sqrt(uev ** 2 + vev ** 2))

    @staticmethod
    def minmod(a, b):
        return torch.where(a * b > 0, torch.where(a > 0, torch.minimum(a, b), torch.maximum(a, b)), 0.0)

    def lowest(self, offsets):
        """Smallest water depth measure over the stencil: min zs + min zb."""
        z = b = None
        for o in offsets:
            p, q = self.at(self.zs, *o), self.at(self.zb, *o)
            z, b = (p, q) if z is None else (torch.minimum(z, p), torch.minimum(b, q))
        return z + b > 2 * self.eps

    def correct(self, dt, u, v, hum, hvm):
        """Second-order corrections of the advected velocities."""
        at, qx, qy, uo, vo, mm, dx = self.at, self.qx, self.qy, self.uuold, self.vvold, self.minmod, self.dx
        inx = torch.ones_like(u, dtype=torch.bool)
        inx[:, 0] = False
        iny = inx.clone()
        iny[0] = False
        inv = iny.clone()
        inv[-2:] = False

        def flux(q, plus, minus, ok):
            return torch.where(ok, torch.where(q > 0, 0.5 * plus, torch.where(q < 0, -0.5 * minus, 0.0)), 0.0)

        a1 = flux(qx + at(qx, -1), mm(u - at(uo, -1), at(u, -1) - at(uo, -2)), mm(uo - at(u, -1), at(uo, 1) - u),
                  inx & self.lowest([(k, 0) for k in (-2, -1, 0, 1, 2)]))
        a2 = flux(at(qy, 1) + qy, mm(at(u, 0, 1) - uo, u - at(uo, 0, -1)), mm(at(uo, 0, 1) - u, at(uo, 0, 2) - at(u, 0, 1)),
                  iny & self.lowest([(i, j) for i in (0, 1) for j in (-1, 0, 1, 2)]))
        b1 = flux(qy + at(qy, 0, -1), mm(v - at(vo, 0, -1), at(v, 0, -1) - at(vo, 0, -2)), mm(vo - at(v, 0, -1), at(vo, 0, 1) - v),
                  inv & self.lowest([(0, k) for k in (-2, -1, 0, 1, 2)]))
        b2 = flux(at(qx, 0, 1) + qx, mm(at(v, 1) - vo, v - at(vo, -1)), mm(at(vo, 1) - v, at(vo, 2) - at(v, 1)),
                  inv & self.lowest([(i, j) for i in (-1, 0, 1, 2) for j in (0, 1)]))
        qe, qw = 0.5 * (at(qx, 1) + qx), 0.5 * (qx + at(qx, -1))
        qn, qs = 0.5 * (at(qy, 0, -1) + at(qy, 1, -1)), 0.5 * (qy + at(qy, -1))
        self.uu = torch.where(iny, u - dt / hum * ((qe * at(a1, 1) - qw * a1) / dx + (qs * a2 - qn * at(a2, 0, -1)) / dx), u)
        qe, qw = 0.5 * (at(qx, 0, 1) + qx), 0.5 * (at(qx, -1) + at(qx, -1, 1))
        qn, qs = 0.5 * (qy + at(qy, 0, -1)), 0.5 * (at(qy, 0, 1) + qy)
        self.vv = torch.where(iny, v - dt / hvm * ((qe * b2 - qw * at(b2, -1)) / dx + (qs * at(b1, 0, 1) - qn * b1) / dx), v)

    def levels(self, dt):
        """Continuity and the second-order water-level correction."""
        at, u, v, zo, mm, dx = self.at, self.uu, self.vv, self.zsold, self.minmod, self.dx
        qx, qy = u * self.hu, v * self.hv
        dz = (at(qx, -1) - qx + at(qy, 0, -1) - qy) / dx
        dz[:, 0] = 0.0
        self.dzsdt = torch.cat([self.dzsdt[:, :1], dz[:, 1:]], 1)
        z = self.zs = self.zs + dz * dt
        inx = torch.ones_like(z, dtype=torch.bool)
        inx[:, 0] = False
        iny = inx.clone()
        iny[0] = False
        w1 = torch.where(u > 0, 0.5 * u * mm(at(z, 1) - zo, z - at(zo, -1)), -0.5 * u * mm(at(zo, 2) - at(z, 1), at(zo, 1) - z))
        w1 = torch.where(inx & self.lowest([(k, 0) for k in (-1, 0, 1, 2)]), w1, 0.0)
        w2 = torch.where(v > 0, 0.5 * v * mm(at(z, 0, 1) - zo, z - at(zo, 0, -1)), 0.5 * v * mm(at(zo, 0, 2) - at(z, 0, 1), at(zo, 0, 1) - z))
        w2 = torch.where(iny & self.lowest([(0, k) for k in (-1, 0, 1, 2)]), w2, 0.0)
        zn = torch.where(iny, z - dt * ((w1 - at(w1, -1)) / dx + (w2 - at(w2, 0, -1)) / dx), z)
        self.zs = self.rows(zn)
        self.qx, self.qy = torch.where(iny, qx + w1, qx), torch.where(iny, qy + w2, qy)
        self.hh = (self.zb + self.zs).clamp(min=self.eps)

    def sediment(self, dt):
        at, dx, g, rho, h = self.at, self.dx, self.g, self.rho, self.hh
        por, D50, D90, wws, morfac = 0.4, 0.00025, 0.00053, 0.0509, self.c.get("morfac", 1.0)
        # wave skewness and asymmetry
        kk = 2 * PI / (self.cc * TREP)
        Ur = (0.375 * math.sqrt(2.0) * self.H * kk / (kk * h) ** 3).clamp(min=1e-5)
        Bm = 0.7939 / (1 + math.exp(-0.6065 / 0.3539) * Ur ** (-math.log10(math.e) / 0.3539))
        B1 = (-90 + 90 * torch.tanh(0.6373 / Ur ** 0.5995)) * PI / 180
        ua = 0.2 * Bm * (torch.cos(B1) - torch.sin(B1)) * self.urms
        ct, st = torch.cos(self.thetamean), torch.sin(self.thetamean)
        ax, ay = 0.5 * (ua + at(ua, 1)), 0.5 * (ua + at(ua, 0, 1))
        urep, vrep = self.ueu + ct * ax, self.vev + st * ay
        mu = torch.sqrt((self.uu + ct * ax) ** 2 + (self.vu + st * ax) ** 2)
        mv = torch.sqrt((self.uv + ct * ay) ** 2 + (self.vv + st * ay) ** 2)
        C, zb = self.C, self.zb
        Cr, Ct = at(C, 1), at(C, 0, 1)
        cu = torch.where(urep > 0, C, torch.where(urep < 0, Cr, 0.5 * (C + Cr)))
        cv = torch.where(vrep > 0, C, torch.where(vrep < 0, Ct, 0.5 * (C + Ct)))
        Dc = self.nuh + h * (self.DR / rho) ** (1 / 3)
        Su = (cu * urep - Dc * (Cr - C) / dx + 1.6 * cu * mu * (at(zb, 1) - zb) / dx) * self.hu * (self.hu > self.eps)
        Sv = (cv * vrep - Dc * (Ct - C) / dx + 1.6 * cv * mv * (at(zb, 0, 1) - zb) / dx) * self.hv * (self.hv > self.eps)
        # equilibrium concentration
        drho = (2650.0 - rho) / rho
        hi = h.clamp(min=0.01)
        vm = (0.5 * (at(self.ueu, -1) + self.ueu)) ** 2 + (0.5 * (at(self.vev, 0, -1) + self.vev)) ** 2
        ML = torch.minimum(torch.sqrt(2 * self.R * TREP / (rho * self.cc)), hi).clamp(min=0.01)
        dcf = (1 / (torch.exp(hi.clamp(max=100.0) / ML) - 1)).clamp(max=1.0)
        Ur2 = self.urms ** 2 + 1.45 * (self.DR / rho) ** (2 / 3) * dcf
        Ts = (0.1 * hi / wws).clamp(min=0.5)
        Ucr = 0.19 * D50 ** 0.1 * torch.log10(4 * hi / D90)
        Cd = (0.4 / (torch.log(hi.clamp(min=0.06) / 0.006) - 1)) ** 2
        de = (drho * g) ** (1 / 3) / 1e-4 * D50
        T1 = torch.sqrt((vm + 0.018 / Cd * Ur2).clamp(max=100000.0 * g / 0.01 * D50 * drho))
        T2 = torch.where((T1 > Ucr) & (hi > self.eps), (T1 - Ucr).clamp(min=0.0) ** 2.4, 0.0)
        Asb = 0.005 * hi * (1 / hi / (drho * g)) ** 1.2
        Ass = 0.012 * D50 * de ** -0.6 / (drho * g * D50) ** 1.2
        wz = (hi > self.eps).double()
        ceq = ((Ass * T2 / hi).clamp(max=0.05) + (Asb * T2 / hi).clamp(max=0.05)) * wz
        fe = (self.stdep / (morfac * dt / (1 - por) * h * ceq / Ts).clamp(min=1e-6)).clamp(max=1.0)
        ero = fe * h * ceq / Ts
        div = (Su - at(Su, -1)) / dx + (Sv - at(Sv, 0, -1)) / dx
        cs = dt * Ts / (dt + Ts) * (h * C / dt - (div - ero)) * wz
        cs = torch.minimum(cs.clamp(min=0.0), 0.1 * h)
        Cn = self.rows(cs / h)
        Cn[:, 0] = 0.0
        self.C = Cn
        dzg = morfac * dt / (1 - por) * (ero - cs / Ts)

        def bed(d):  # the bed's boundary rule
            e = self.rows(d)
            e[:, 0] = d[:, 1]
            return e

        def take(a, d):  # value and change of the source cell
            return bed(a) + bed(d)

        hb = h + dzg
        zb, sd = take(zb, dzg), take(self.stdep, -dzg)
        # avalanching
        lim = torch.where(hb > self.eps, 0.3, 1.0)

        def exchange(ax):
            A = lambda f: at(f, 1) if ax == 0 else at(f, 0, 1)  # noqa: E731
            s = (A(zb) - zb) / dx
            b = torch.sign(s) * (s.abs() - lim) * dx
            up = torch.minimum(torch.minimum(b, torch.full_like(b, 0.01 * dt / dx)), sd)
            dn = torch.maximum(torch.maximum(b, torch.full_like(b, -0.01 * dt / dx)), -A(sd))
            return torch.where(s.abs() > lim, torch.where(s > 0, up, dn), 0.0)

        ex, ey = exchange(0), exchange(1)
        d = ex + ey
        d[:, 1:] -= ex[:, :-1]
        d[1:] -= ey[:-1]
        self.zs, self.hh = self.zs - d, hb - d
        self.zb, self.stdep = take(zb, d), take(sd, -d)


def _net(P, x, t=None):
    """The surrogate in float64, its parameters rounded as the network holds
    them: outputs, or loss and gradients in the order of the parameters."""
    prm, o = [], 0
    for cin, cout, taps, _ in SUR:
        w = P[o:o + taps * cout * cin].double().reshape(taps, cout, cin)
        o += taps * cout * cin
        b = P[o:o + cout].double()
        o += cout
        prm.append([w.to(x.device).requires_grad_(t is not None), b.to(x.device).requires_grad_(t is not None)])

    def conv(l, v):
        w, b = prm[l]
        n, H, W, cin = v.shape
        if w.shape[0] == 1:
            y = v.reshape(-1, cin) @ w[0].T + b
            y = y.reshape(n, H, W, -1)
        else:
            vp = F.pad(v, (0, 0, 1, 1, 1, 1))
            y = b
            for k in range(9):
                s = vp[:, k // 3:k // 3 + H, k % 3:k % 3 + W].reshape(-1, cin)
                y = y + (s @ w[k].T).reshape(n, H, W, -1)
        return torch.relu(y) if SUR[l][3] else y

    def pool(v):
        return 0.25 * (v[:, ::2, ::2] + v[:, ::2, 1::2] + v[:, 1::2, ::2] + v[:, 1::2, 1::2])

    def up(v):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2)

    v = F.pad(x.double(), (0, 24))
    e0 = conv(1, conv(0, v))
    e1 = conv(3, conv(2, pool(e0)))
    e2 = conv(5, conv(4, pool(e1)))
    v = conv(8, conv(7, conv(6, pool(e2))))
    v = conv(11, conv(10, conv(9, torch.cat([up(v), e2], -1))))
    v = conv(14, conv(13, conv(12, torch.cat([up(v), e1], -1))))
    y = conv(17, conv(16, conv(15, torch.cat([up(v), e0], -1))))
    if t is None:
        return y
    loss = ((y - t.double()) ** 2).mean()
    loss.backward()
    g = torch.cat([q.grad.reshape(-1).cpu() for p in prm for q in p])
    return dict(loss=float(loss), grads=g.numpy())


def exact(case, seed):
    c = case
    if c["kind"] == "step":
        m = _Model(c, seed)
        dt = m.next_dt(T0 + 1.0, 0.1)
        t = T0 + 1.0 + dt
        m.step(t, dt)
        return dict({k: getattr(m, k) for k in STEP_OUT}, t=t, dt=dt)
    if c["kind"] == "window":
        m = _Model(c, seed)
        m.products(_products(c, seed))
        t, dt, n, stop = T0 + 1.0, 0.1, 0, T0 + 1.0 + c["seconds"]
        mean = dict(uumean=0.0, vvmean=0.0, zsmean=0.0, Hmean=0.0)
        while t < stop:
            dt = m.next_dt(t, dt, stop, with_wave=False)
            t += dt
            m.step(t, dt, wave=False)
            n += 1
            for k in mean:
                mean[k] = mean[k] + getattr(m, k[:-4])
        out = {k: getattr(m, k) for k in ("zs", "uu", "vv", "hh", "zb", "C")}
        return dict(out, **{k: v / n for k, v in mean.items()}, n=n, dt=dt)
    if c["kind"] == "ensemble":
        parts = []
        for k, d in enumerate(_ensemble_cases(c)):
            m = _Model(d, seed * 1000 + k)
            t, dt = T0 + 1.0, 0.1
            acc = None
            for _ in range(c["steps"]):
                dt = m.next_dt(t, dt, 1e9)
                t += dt
                m.step(t, dt)
                v = torch.stack([m.zs, m.uu, m.vv, m.H, m.Dw, m.DR, m.Fx, m.Fy], -1)
                acc = v if acc is None else acc + v
            acc = acc / c["steps"]
            sea = torch.tensor([d["Hm0"], 10.0, math.radians(d["dir"])], dtype=torch.float64, device=acc.device)
            parts.append(torch.cat([m.zb[..., None], acc[..., :3], sea.expand(d["ny"], d["nx"], 3), acc[..., 3:]], -1).reshape(-1))
        return torch.cat(parts)
    P, f, sea, x, t5 = _sur_inputs(c, seed)
    if c["kind"] == "infer":
        v = torch.cat([f.permute(0, 2, 3, 1).double(), sea.double()[:, None, None, :].expand(c["n"], c["H"], c["W"], 3)], -1)
        n14 = torch.tensor(NORM14, device=v.device).double()
        v = F.pad((v - n14[:7]) / n14[7:], (0, 1))
        with torch.no_grad():
            return _net(P, v)
    return _net(P, x, t5)
