"""Timed cases: the calls a user's program makes of this package, over the sizes it is used at.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` builds
what a program holds before the call (a solver with its fields, an ensemble, a network with
its batch), ``run`` makes one pass through the public entry points, ``work`` states the bytes
and operations a pass cannot do without, and ``exact`` states the same pass in plain torch
FP64, independently of the library.

What the kinds stand for in use:

* ``dns``       a flow advanced ``steps`` time steps, as ``tcsolver`` and a driver script do:
                ``sync`` steps one by one and takes dt back after each (integrate()), otherwise
                the steps are queued; ``logged`` also reads the energy diagnostics and adds a
                statistics sample after them, as the log and statistics schedules do;
* ``ensemble``  many uneven flows advanced together, replayed from recorded graphs;
* ``closure``   the coarse solver with the learned closure coupled;
* ``train``     one Adam step of the closure network on a host batch;
* ``predict``   the network evaluated on a host batch (validation, the closure's power).

The results of a flow are the solver's own device buffers: ``run`` returns a dict whose
entries are copied to the host when they are looked up, since a program that steps a flow
reads its fields only now and then.
"""
import math
import random

import numpy as np
import torch

import simpletcsolver_amd as tc

GAMMA = (32. / 60., 8. / 60., 20. / 60.)
ALPHA = (32. / 60., 25. / 60., 45. / 60.)
BETA = (0., -17. / 60., -25. / 60.)
VELOCITY = ("ux", "uy", "uz")
UY_WALLS = (1.0, 0.0)
T_WALLS = (0.5, -0.5)
# flows of more cells than this start from the library's own seeded fields, made on the
# device; smaller ones from fields of the caller, as a restart from a checkpoint does
MOST_HOST_CELLS = 10_000_000


def _dns(name, nx, ny, nz, implicit, steps, curved=True, Re=1000.0, scalar=True, stretch=2.0,
         precision="fp64", sync=False, logged=False, dt_fixed=0.0, eta=0.714):
    return dict(name=name, kind="dns", nx=nx, ny=ny, nz=nz, curved=curved, Re=Re, implicit=implicit,
                scalar=scalar, stretch=stretch, precision=precision, steps=steps, sync=sync,
                logged=logged, dt_fixed=dt_fixed, eta=eta)


def listed():
    return [
        # the reference's documented example (Re = 80), stepped one by one: all latency
        _dns("typical_64x8x32", 64, 8, 32, "x", 1, Re=80.0, stretch=1.0, sync=True, eta=0.5),
        # the smallest benchmark configuration: explicit, fixed step, no scalar
        _dns("explicit_64x64x64", 64, 64, 64, "", 10, scalar=False, stretch=1.0, dt_fixed=1e-3),
        # a channel of ragged sizes with transform lengths of every radix, all diffusion implicit
        _dns("ragged_97x150x105", 97, 150, 105, "xyz", 5, curved=False),
        # a production run with its log and statistics samples
        _dns("logged_128x192x256", 128, 192, 256, "x", 4, Re=2000.0, sync=True, logged=True),
        # the middle benchmark configuration
        _dns("dns_256x512x512", 256, 512, 512, "x", 2, Re=5000.0),
        # mixed precision, and its refined form at odd sizes
        _dns("mixed_256x512x512", 256, 512, 512, "xyz", 2, Re=5000.0, precision="mixed"),
        _dns("refined_150x140x180", 150, 140, 180, "xyz", 4, precision="mixed_refined"),
        # the headline configuration
        _dns("dns_512x1024x1024", 512, 1024, 1024, "xyz", 1, Re=1e4),
        # a parameter sweep of uneven flows (the ensemble benchmark's ranges, a quarter of it)
        dict(name="ensemble_16", kind="ensemble", members=16, pick=7, steps=4),
        # the closure's coarse run, its training and its evaluation
        dict(name="closure_32x64x64", kind="closure", nx=32, ny=64, nz=64, Re=3000.0, steps=10),
        dict(name="train_32x64x64", kind="train", nx=32, ny=64, nz=64, batch=4),
        dict(name="predict_64x128x128", kind="predict", nx=64, ny=128, nz=128, batch=1),
    ]


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_size(rng, lo, hi, even):
    """a length the transforms take (2, 3, 5 and 7 as factors), spread over the logarithm"""
    while True:
        n = _size(rng, lo, hi)
        m = 2 * max(2, n // 2) if even else n
        if lo <= m <= hi and _smooth(m // 2 if even else m):
            return m


def draw(rng):
    kind = rng.choice(("dns", "dns", "dns", "dns", "mixed", "mixed_refined", "ensemble", "closure", "train", "predict"))
    if kind in ("dns", "mixed", "mixed_refined"):
        while True:
            nx, ny, nz = _size(rng, 24, 640), _smooth_size(rng, 8, 1024, True), _smooth_size(rng, 12, 1024, False)
            if nx * ny * nz <= 1 << 28:
                break
        steps = max(1, min(10, 20_000_000 // (nx * ny * nz)))
        implicit = rng.choice(("", "x", "x", "xy", "xyz", "xyz"))
        logged = rng.random() < 0.15
        return dict(kind="dns", nx=nx, ny=ny, nz=nz, curved=rng.random() < 0.8, Re=float(round(_size(rng, 80, 10000))),
                    implicit=implicit, scalar=rng.random() < 0.7, stretch=1.0 if implicit == "" else 2.0,
                    precision="fp64" if kind == "dns" else kind, steps=steps,
                    sync=logged or rng.random() < 0.25, logged=logged, dt_fixed=0.0)
    if kind == "ensemble":
        return dict(kind="ensemble", members=rng.randint(4, 24), pick=rng.randint(0, 10 ** 6), steps=rng.randint(1, 4))
    nx, ny, nz = _size(rng, 24, 80), _smooth_size(rng, 32, 128, True), _smooth_size(rng, 32, 128, False)
    if kind == "closure":
        return dict(kind="closure", nx=nx, ny=ny, nz=nz, Re=float(_size(rng, 1000, 10000)), steps=10)
    batch = rng.randint(1, 8)
    while nx * ny * nz * batch > 1 << 20:
        batch = max(1, batch // 2)
        nz = nz if batch > 1 else _smooth_size(rng, 32, 64, False)
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, batch=batch)


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _grid(nx, lx, curved, stretch):
    """tanh-clustered faces xf (nx+1) and centres xc (nx+2)"""
    ri = 1.0 if curved else 0.0
    s = 2.0 * np.arange(nx + 1) / nx - 1.0
    xf = ri + 0.5 * lx * (1.0 + np.tanh(stretch * s) / math.tanh(stretch))
    xf[0], xf[nx] = ri, ri + lx
    xc = np.concatenate([xf[:1], 0.5 * xf[:-1] + 0.5 * xf[1:], xf[-1:]])
    return xf, xc


def _setup(case):
    """grid and Solver arguments of a flow"""
    eta = case.get("eta", 0.714)
    lx = 1.0 / eta - 1.0 if case["curved"] else 1.0
    lengths = (lx, math.pi / 3.0, 2.0 * math.pi * lx) if case["curved"] else (1.0, 1.0, 2.0)
    xf, xc = _grid(case["nx"], lx, case["curved"], case["stretch"])
    kw = dict(is_curved=case["curved"], lengths=lengths, Re=case["Re"],
              implicit=tuple(int(d in case["implicit"]) for d in "xyz"), scalar=int(case["scalar"]),
              uy_walls=UY_WALLS, t_walls=T_WALLS, coef_dt_adv=0.5, coef_dt_dif=0.5,
              dt_fixed=case.get("dt_fixed", 0.0), precision=case.get("precision", "fp64"))
    return xf, xc, kw


def _fields(case, seed):
    """a perturbed laminar flow in the NPY layout: the wall-driven profile, four modes per
    direction and a little noise; T the conduction profile, p zero"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    xf, xc, _ = _setup(case)
    rng = np.random.default_rng(seed)
    ri, ro = xf[0], xf[-1]
    y, z = np.arange(ny) / ny, np.arange(nz) / nz

    def modes(x):
        xi = (x - ri) / (ro - ri)
        a = np.zeros((nz, ny, len(x)))
        for m in range(1, 5):
            w, py, pz = rng.uniform(-1, 1), rng.uniform(0, 2 * np.pi), rng.uniform(0, 2 * np.pi)
            a += (0.05 * w * np.sin(np.pi * m * xi)[None, None, :] * np.cos(2 * np.pi * m * y + py)[None, :, None]
                  * np.cos(2 * np.pi * m * z + pz)[:, None, None])
        a[..., 1:-1] += 1e-3 * rng.uniform(-1, 1, (nz, ny, len(x) - 2))
        return a

    f = {"ux": modes(xf), "uy": modes(xc), "uz": modes(xc)}
    f["ux"][..., [0, -1]] = 0.0
    if case["curved"]:
        a = (UY_WALLS[1] * ro - UY_WALLS[0] * ri) / (ro * ro - ri * ri)
        b = ri * ro * (UY_WALLS[0] * ro - UY_WALLS[1] * ri) / (ro * ro - ri * ri)
        f["uy"] += a * xc + b / xc
    else:
        f["uy"] += UY_WALLS[1] + (UY_WALLS[0] - UY_WALLS[1]) * (ro - xc) / (ro - ri)
    f["t"] = np.broadcast_to(T_WALLS[1] + (T_WALLS[0] - T_WALLS[1]) * (ro - xc) / (ro - ri), (nz, ny, nx + 2)).copy()
    f["t"][..., 1:-1] += 1e-2 * rng.uniform(-1, 1, (nz, ny, nx))
    f["p"] = np.zeros((nz, ny, nx + 2))
    for n, w in (("uy", UY_WALLS), ("uz", (0.0, 0.0)), ("t", T_WALLS)):
        f[n][..., 0], f[n][..., -1] = w
    return f


def _member_cases(case):
    """the ensemble's flows: the ranges of the ensemble benchmark"""
    rng = random.Random(case["pick"])
    out = []
    for _ in range(case["members"]):
        curved = rng.random() >= 0.1
        out.append(dict(nx=rng.randint(64, 128), ny=rng.choice((128, 192, 256)), nz=rng.choice((128, 192, 256)),
                        curved=curved, eta=rng.uniform(0.5, 0.9), Re=float(rng.randint(500, 8000)), implicit="",
                        scalar=False, stretch=1.0))
    return out


def _layers(seed):
    """He-normal weights [27][co][ci] and small biases; rows past the 5 input and 4 output
    channels in use are zero"""
    rng = np.random.default_rng(seed + 1000)
    out = []
    for l, (taps, co, ci) in enumerate(tc.CNN_SHAPES):
        w = rng.standard_normal((taps, co, ci)) * math.sqrt(2.0 / (27 * (5 if l == 0 else ci))) * (0.1 if l == 2 else 1.0)
        b = 0.05 * rng.standard_normal(co)
        if l == 0:
            w[:, :, 5:] = 0.0
        if l == 2:
            w[:, 4:, :] = 0.0
            b[4:] = 0.0
        out.append((w.astype(np.float32), b.astype(np.float32)))
    return out


def _batch(case, seed):
    """normalised inputs and targets of a training set: unit variance, smooth plus noise"""
    rng = np.random.default_rng(seed)
    shape = (case["batch"], case["nz"], case["ny"], case["nx"])
    x = rng.standard_normal(shape + (5,), dtype=np.float32)
    y = rng.standard_normal(shape + (4,), dtype=np.float32)
    phase = (np.arange(case["nx"]) / case["nx"] * 2 * np.pi).astype(np.float32)
    x = (0.8 * x + 0.6 * np.sqrt(np.float32(2)) * np.sin(phase)[:, None]).astype(np.float32)
    return x, y


def _closure_norm():
    mean = np.array([0.0, 0.4, 0.0, 0.0, 1.2], dtype=np.float32)
    std = np.array([0.05, 0.3, 0.05, 0.3, 0.12], dtype=np.float32)
    scale = np.array([1e-2, 1e-2, 1e-2, 1e-2], dtype=np.float32)
    return mean, std, scale


# ------------------------------------------------------------------------------------------
# results read from the device when they are looked up
# ------------------------------------------------------------------------------------------
class Results(dict):
    def __init__(self, keep, **readers):
        super().__init__(readers)
        self._keep = keep   # the objects whose buffers these are

    def __getitem__(self, key):
        v = super().__getitem__(key)
        return v() if callable(v) else v


def _no_gauge(p):
    """the pressure without its free constant: it is determined up to a constant only, which
    the singular radial mode leaves to rounding"""
    return p - p.mean()


def _field_reader(flows, name, scalar):
    def read():
        got = [(_no_gauge(s.get_field(name)) if name == "p" else s.get_field(name)) for s in flows]
        return got[0] if len(got) == 1 else np.concatenate([a.ravel() for a in got])
    return read


def _flow_results(state, flows, scalar, **more):
    names = VELOCITY + (("p", "t") if scalar else ("p",))
    return Results(state, dt=lambda: np.array([s.dt() for s in flows]),
                   **{n: _field_reader(flows, n, scalar) for n in names}, **more)


# ------------------------------------------------------------------------------------------
# prepare and run
# ------------------------------------------------------------------------------------------
def _solver(case, seed):
    xf, xc, kw = _setup(case)
    s = tc.Solver(case["nx"], case["ny"], case["nz"], xf, xc, **kw)
    if case["nx"] * case["ny"] * case["nz"] > MOST_HOST_CELLS:
        s.ic(seed=seed + 1, amp=1e-3, t_amp=1e-2, nmodes=4, mode_amp=0.1)
    else:
        s.load_fields(_fields(case, seed))
    return s


def _closure_case(case):
    return dict(case, curved=True, implicit="x", scalar=True, stretch=2.0, dt_fixed=0.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dns":
        s = _solver(case, seed)
        if case["logged"]:
            s.arm_diagnostics(True)
            s.stat_arm(True)
        return dict(case=case, flow=s)
    if kind == "ensemble":
        specs, members = [], _member_cases(case)
        for m in members:
            xf, xc, kw = _setup(m)
            specs.append(dict(nx=m["nx"], ny=m["ny"], nz=m["nz"], xf=xf, xc=xc, **kw))
        e = tc.Ensemble(specs)
        for q, s in enumerate(e.members):
            s.ic(seed=100 * seed + q + 1, amp=1e-3, t_amp=0.0, nmodes=4, mode_amp=0.1)
        return dict(case=case, ensemble=e)
    if kind == "closure":
        s = _solver(_closure_case(case), seed)
        net = tc.Cnn(case["nx"], case["ny"], case["nz"], batch=1)
        for l, (w, b) in enumerate(_layers(seed)):
            net.set_layer(l, w, b)
        tc.attach_closure(s, net, *_closure_norm())
        return dict(case=case, flow=s, coupled=net)
    net = tc.Cnn(case["nx"], case["ny"], case["nz"], batch=case["batch"])
    for l, (w, b) in enumerate(_layers(seed)):
        net.set_layer(l, w, b)
    x, y = _batch(case, seed)
    return dict(case=case, net=net, x=x, y=y)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dns":
        s = state["flow"]
        if case["sync"]:
            for _ in range(case["steps"]):
                s.step()
        else:
            s.step_async(case["steps"])
        more = {}
        if case["logged"]:
            more = dict(injection=s.injection(), dissipation=s.dissipation(), energy=s.total_energy())
            s.stat_collect()
            more["stats"] = lambda: s.stats()[0]
        return _flow_results(state, [s], case["scalar"], **more)
    if kind == "ensemble":
        e = state["ensemble"]
        e.step(case["steps"])
        return _flow_results(state, e.members, False)
    if kind == "closure":
        s = state["flow"]
        s.step_async(case["steps"])
        return _flow_results(state, [s], True)
    net = state["net"]
    if kind == "train":
        loss = net.train_step(state["x"], state["y"], 1e-3)
        return Results(state, loss=loss, layers=lambda: [net.layer(l) for l in range(3)])
    return net.predict(state["x"])


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        parts = [work(dict(m, kind="dns", steps=case["steps"])) for m in _member_cases(case)]
        return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}
    cells = case["nx"] * case["ny"] * case["nz"] * case.get("batch", 1)
    # multiply-adds of the three layers per cell: 27 taps of 5 x 32, 32 x 32 and 32 x 4 channels
    macs = 27 * (5 * 32 + 32 * 32 + 32 * 4)
    if kind == "predict":
        return {"bytes": cells * 4 * (5 + 4), "flops": 2 * macs * cells}
    if kind == "train":
        # forward, the weights' gradients, and the data gradients of the last two layers
        return {"bytes": cells * 4 * (5 + 4), "flops": 2 * cells * (2 * macs + 27 * (32 * 32 + 32 * 4))}
    if kind == "closure":
        case = _closure_case(case)
    # a step: the state (velocity, scalar, pressure) in and out; right-hand sides, transforms
    # and line solves of three substeps
    nf = 4 if case["scalar"] else 3
    rhs = 110 * nf
    fft = 2 * (2.5 * math.log2(case["ny"]) + 5 * math.log2(case["nz"]))
    solves = 8 * nf * len(case["implicit"]) + 16
    flops = 3 * cells * (rhs + fft + solves + 40)
    if kind == "closure":
        flops += 2 * macs * cells
    return {"bytes": case["steps"] * cells * 8 * 2 * (nf + 1), "flops": case["steps"] * flops}


# ------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _yp(a):
    return torch.roll(a, -1, 1)


def _ym(a):
    return torch.roll(a, 1, 1)


def _zp(a):
    return torch.roll(a, -1, 0)


def _zm(a):
    return torch.roll(a, 1, 0)


def _flux(am, ap, qm, q, qp, j):
    """- (1/J) of the advective flux difference in skew-symmetric form"""
    return -(0.5 * ap * (qp - q) + 0.5 * am * (q - qm)) / j


def _thomas(l, c, u, d):
    """tridiagonal systems along the last axis; l, c, u broadcast against d"""
    n = d.shape[-1]
    c = c.expand(d.shape) if c.dim() == d.dim() else c
    v, q = [u[..., 0] / c[..., 0]], [d[..., 0] / c[..., 0]]
    for i in range(1, n):
        r = 1.0 / (c[..., i] - l[..., i] * v[-1])
        v.append(r * u[..., i])
        q.append(r * (d[..., i] - l[..., i] * q[-1]))
    for i in range(n - 2, -1, -1):
        q[i] = q[i] - v[i] * q[i + 1]
    return torch.stack(q, -1)


def _periodic(d, dim, a):
    """(1 - a second difference) x = d, periodic along dim; a per radial position or a number"""
    n = d.shape[dim]
    lam = 2.0 - 2.0 * torch.cos(2.0 * math.pi * torch.arange(n, device=d.device, dtype=torch.float64) / n)
    lam = lam.reshape((n, 1, 1) if dim == 0 else (1, n, 1))
    return torch.fft.ifft(torch.fft.fft(d, dim=dim) / (1.0 + a * lam), dim=dim).real


class _Flow:
    """one flow, array layout (z, y, x): ux at the faces, the others at the centres with the
    two wall values"""

    def __init__(self, case, fields):
        xf, xc, kw = _setup(case)
        t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_device())  # noqa: E731
        self.nx, self.ny, self.nz = case["nx"], case["ny"], case["nz"]
        self.kw = kw
        self.f = {n: t(fields[n]) for n in ("ux", "uy", "uz", "p", "t")}
        xf, xc = t(xf), t(xc)
        self.hxf = xc[1:] - xc[:-1]
        self.hxc = torch.cat([0.5 * (xf[1:2] - xf[:1]), xf[1:] - xf[:-1], 0.5 * (xf[-1:] - xf[-2:-1])])
        ly = kw["lengths"][1] / self.ny
        self.hyf = xf * ly if case["curved"] else torch.full_like(xf, ly)
        self.hyc = xc * ly if case["curved"] else torch.full_like(xc, ly)
        self.hz = kw["lengths"][2] / self.nz
        self.jf, self.jc = self.hxf * self.hyf * self.hz, self.hxc * self.hyc * self.hz
        self.nu = self.kappa = 1.0 / case["Re"]
        self.old = {}
        self.extra = None

    def dt(self):
        if self.kw["dt_fixed"] > 0:
            return self.kw["dt_fixed"]
        u, v, w = self.f["ux"], self.f["uy"][..., 1:-1], self.f["uz"][..., 1:-1]
        adv = min(1.0, float((self.hxf[1:-1] / (u[..., 1:-1].abs() + 1e-8)).min()),
                  float((self.hyc[1:-1] / (v.abs() + 1e-8)).min()), float((self.hz / (w.abs() + 1e-8)).min()))
        out = adv * self.kw["coef_dt_adv"]
        grid = (float(self.hxc.min()), float(self.hyc[1]), self.hz)
        for d in range(3):
            if not self.kw["implicit"][d]:
                out = min(out, self.kw["coef_dt_dif"] / max(self.nu, self.kappa) * 0.5 / 3.0 * grid[d] ** 2)
        return out

    def tensors(self):
        """gradients on the staggered grid: the face-centred ones at faces 1..nx+1"""
        U, V, W = self.f["ux"], self.f["uy"], self.f["uz"]
        df = self.jc[1:] / self.hxc[1:] - self.jc[:-1] / self.hxc[:-1]
        mx = self.jf / self.hxf
        dc = mx[1:] - mx[:-1]
        wl, wr = torch.full_like(self.jf, 0.5), torch.full_like(self.jf, 0.5)
        wl[0] = wr[-1] = 0.0
        g = {}
        g["lyx0"] = (U - _ym(U)) / self.hyf
        g["lyx1"] = -df / self.jf * (wl * V[..., :-1] + wr * V[..., 1:])
        g["lxy"] = (V[..., 1:] - V[..., :-1]) / self.hxf
        g["lxz"] = (W[..., 1:] - W[..., :-1]) / self.hxf
        g["lxx"] = (U[..., 1:] - U[..., :-1]) / self.hxc[1:-1]
        v, w = V[..., 1:-1], W[..., 1:-1]
        g["lyy0"] = (_yp(v) - v) / self.hyc[1:-1]
        g["lyy1"] = dc / self.jc[1:-1] * 0.5 * (U[..., :-1] + U[..., 1:])
        g["lyz"] = (w - _ym(w)) / self.hyc[1:-1]
        g["lzx"] = (U - _zm(U)) / self.hz
        g["lzy"] = (v - _zm(v)) / self.hz
        g["lzz"] = (_zp(w) - w) / self.hz
        return g

    def rhs(self, g):
        """explicit (a) and trapezoidal (g) right-hand sides of the advected fields"""
        U, V, W, P, T = (self.f[n] for n in ("ux", "uy", "uz", "p", "t"))
        jf, jc, hxf, hxc, hyc, hz, nu = self.jf, self.jc, self.hxf, self.hxc, self.hyc, self.hz, self.nu
        imp = self.kw["implicit"]
        I = slice(1, -1)  # noqa: E741
        mx = jf / hxf
        dc = mx[1:] - mx[:-1]
        df = jc[1:] / hxc[1:] - jc[:-1] / hxc[:-1]
        fx, fy, fz = mx * U, jc / hyc * V, jc / hz * W
        out = {}

        def split(name, a, dif, gp):
            gg = gp
            for d in range(3):
                if imp[d]:
                    gg = gg + dif[d]
                else:
                    a = a + dif[d]
            if self.extra is not None:
                a = a + self.extra[name]
            out[name] = (a, gg)

        # ux at the interior faces
        j, q = jf[I], U[..., I]
        fxc = 0.5 * (fx[..., :-1] + fx[..., 1:])
        fyf, fzf = 0.5 * (fy[..., :-1] + fy[..., 1:])[..., I], 0.5 * (fz[..., :-1] + fz[..., 1:])[..., I]
        a = _flux(fxc[..., :-1], fxc[..., 1:], U[..., :-2], q, U[..., 2:], j)
        a = a + _flux(fyf, _yp(fyf), _ym(q), q, _yp(q), j) + _flux(fzf, _zp(fzf), _zm(q), q, _zp(q), j)
        vc = 0.5 * (V + _yp(V))[..., I]
        c = dc * vc * vc
        a = a + 0.5 * (c[..., :-1] + c[..., 1:]) / j
        s = (g["lyx1"] + g["lxy"])[..., I]
        a = a + nu * (_yp(s) - s) / self.hyf[I]
        s = g["lxz"][..., I]
        a = a + nu * (_zp(s) - s) / hz
        c = dc * (g["lyy0"] + g["lyy1"])
        a = a - 2.0 * nu * 0.5 * (c[..., :-1] + c[..., 1:]) / j
        s = jc[I] * g["lxx"] / hxc[I]
        dif = [2.0 * nu * (s[..., 1:] - s[..., :-1]) / j, nu * (_yp(q) - 2.0 * q + _ym(q)) / self.hyf[I] ** 2,
               nu * (_zp(q) - 2.0 * q + _zm(q)) / hz ** 2]
        split("ux", a, dif, -((P[..., 1:] - P[..., :-1]) / hxf)[..., I])

        # uy at the centres
        j, q, h = jc[I], V[..., I], hyc[I]
        fxf = 0.5 * (_ym(fx) + fx)
        a = _flux(fxf[..., :-1], fxf[..., 1:], V[..., :-2], q, V[..., 2:], j)
        m = 0.5 * (_ym(fy) + fy)[..., I]
        a = a + _flux(m, _yp(m), _ym(q), q, _yp(q), j)
        m = 0.5 * (_ym(fz) + fz)[..., I]
        a = a + _flux(m, _zp(m), _zm(q), q, _zp(q), j)
        uc = 0.5 * (U[..., :-1] + U[..., 1:])
        m = 0.5 * (_ym(q) + q) * _ym(uc)
        a = a - 0.5 * dc * (m + _yp(m)) / j
        lyx = g["lyx0"] + g["lyx1"]
        s = mx * lyx
        a = a + nu * (s[..., 1:] - s[..., :-1]) / j
        s = g["lyy1"]
        a = a + 2.0 * nu * (s - _ym(s)) / h
        s = g["lyz"]
        a = a + nu * (_zp(s) - s) / hz
        s = df * (lyx + g["lxy"])
        a = a + nu * 0.5 * (s[..., :-1] + s[..., 1:]) / j
        lap = self.laps(V)
        p = P[..., I]
        split("uy", a, [nu * lap[0], 2.0 * nu * lap[1], nu * lap[2]], -(p - _ym(p)) / h)

        # uz at the centres
        q = W[..., I]
        fxf = 0.5 * (_zm(fx) + fx)
        a = _flux(fxf[..., :-1], fxf[..., 1:], W[..., :-2], q, W[..., 2:], j)
        m = 0.5 * (_zm(fy) + fy)[..., I]
        a = a + _flux(m, _yp(m), _ym(q), q, _yp(q), j)
        m = 0.5 * (_zm(fz) + fz)[..., I]
        a = a + _flux(m, _zp(m), _zm(q), q, _zp(q), j)
        s = mx * g["lzx"]
        a = a + nu * (s[..., 1:] - s[..., :-1]) / j
        s = g["lzy"]
        a = a + nu * (_yp(s) - s) / h
        lap = self.laps(W)
        split("uz", a, [nu * lap[0], nu * lap[1], 2.0 * nu * lap[2]], -(p - _zm(p)) / hz)

        if self.kw["scalar"]:
            q = T[..., I]
            a = _flux(fx[..., :-1], fx[..., 1:], T[..., :-2], q, T[..., 2:], j)
            a = a + _flux(fy[..., I], _yp(fy[..., I]), _ym(q), q, _yp(q), j)
            a = a + _flux(fz[..., I], _zp(fz[..., I]), _zm(q), q, _zp(q), j)
            lap = self.laps(T)
            split("t", a, [self.kappa * v for v in lap], torch.zeros_like(q))
        return out

    def laps(self, Q):
        """second differences in x, y and z of a centred field at the interior centres"""
        s = self.jf / self.hxf * (Q[..., 1:] - Q[..., :-1]) / self.hxf
        q = Q[..., 1:-1]
        return [(s[..., 1:] - s[..., :-1]) / self.jc[1:-1], (_yp(q) - 2.0 * q + _ym(q)) / self.hyc[1:-1] ** 2,
                (_zp(q) - 2.0 * q + _zm(q)) / self.hz ** 2]

    def update(self, r, dt, rhs):
        I = slice(1, -1)  # noqa: E741
        fac = {"ux": (2, 1, 1), "uy": (1, 2, 1), "uz": (1, 1, 2), "t": (1, 2, 1)}
        for n, (a, g) in rhs.items():
            d = dt * (ALPHA[r] * a + GAMMA[r] * g)
            if r > 0:
                d = d + dt * BETA[r] * self.old[n]
            pf = 0.5 * GAMMA[r] * dt * (self.kappa if n == "t" else self.nu)
            if self.kw["implicit"][0]:
                if n == "ux":
                    l, u = (self.jc[1:-2] / self.hxc[1:-2] ** 2 / self.jf[I], self.jc[2:-1] / self.hxc[2:-1] ** 2 / self.jf[I])
                else:
                    l, u = (self.jf[:-1] / self.hxf[:-1] ** 2 / self.jc[I], self.jf[1:] / self.hxf[1:] ** 2 / self.jc[I])
                f = fac[n][0] * pf
                d = _thomas(-f * l, 1.0 + f * (l + u), -f * u, d)
            if self.kw["implicit"][1]:
                h = self.hyf[I] if n == "ux" else self.hyc[I]
                d = _periodic(d, 1, fac[n][1] * pf / h ** 2)
            if self.kw["implicit"][2]:
                d = _periodic(d, 0, fac[n][2] * pf / self.hz ** 2)
            self.f[n] = self.f[n].clone()
            self.f[n][..., I] += d
            self.old[n] = a

    def project(self, r, dt):
        I = slice(1, -1)  # noqa: E741
        U, V, W = self.f["ux"], self.f["uy"][..., I], self.f["uz"][..., I]
        jc, hyc, hz, nx, ny, nz = self.jc[I], self.hyc[I], self.hz, self.nx, self.ny, self.nz
        m = self.jf / self.hxf * U
        div = (m[..., 1:] - m[..., :-1]) / jc + (_yp(V) - V) / hyc + (_zp(W) - W) / hz
        s = torch.fft.fft(torch.fft.rfft(div / (GAMMA[r] * dt), dim=1), dim=0)
        k = lambda n, c: (-4.0 * torch.sin(math.pi * torch.arange(c, device=s.device, dtype=torch.float64) / n) ** 2)  # noqa: E731
        l = self.jf[:-1] / self.hxf[:-1] ** 2 / jc
        u = self.jf[1:] / self.hxf[1:] ** 2 / jc
        c = -l - u
        c[0] += l[0]
        c[-1] += u[-1]
        c = c + k(ny, ny // 2 + 1)[None, :, None] / hyc ** 2 + k(nz, nz)[:, None, None] / hz ** 2
        c[0, 0, -1] += 1.0   # the singular mode: any regularisation leaves a constant only
        psi = _thomas(l, c, u, s)
        psi = torch.fft.irfft(torch.fft.ifft(psi, dim=0), n=ny, dim=1)
        psi = torch.cat([psi[..., :1], psi, psi[..., -1:]], -1)
        q, f = psi[..., I], GAMMA[r] * dt
        for n in VELOCITY:
            self.f[n] = self.f[n].clone()
        self.f["ux"][..., I] -= f * (psi[..., 2:-1] - psi[..., 1:-2]) / self.hxf[I]
        self.f["uy"][..., I] -= f * (q - _ym(q)) / hyc
        self.f["uz"][..., I] -= f * (q - _zm(q)) / hz
        p = self.f["p"][..., I] + q
        lap = self.laps(psi)
        for d in range(3):
            if self.kw["implicit"][d]:
                p = p - 2.0 * 0.5 * f * self.nu * lap[d]
        self.f["p"] = torch.cat([p[..., :1], p, p[..., -1:]], -1)

    def step(self):
        dt = self.dt()
        for r in range(3):
            self.stale = self.tensors()
            self.update(r, dt, self.rhs(self.stale))
            self.project(r, dt)
        return dt

    def results(self, dt):
        out = {n: self.f[n].cpu().numpy() for n in VELOCITY}
        out["p"] = _no_gauge(self.f["p"].cpu().numpy())
        if self.kw["scalar"]:
            out["t"] = self.f["t"].cpu().numpy()
        out["dt"] = np.array([dt])
        return out

    def logged(self):
        """energy diagnostics (the gradients those of the last substep's start, the scalar
        the current one) and one statistics sample"""
        g, T = self.stale, self.f["t"]
        jf, jc, hxf, hz = self.jf, self.jc[1:-1], self.hxf, self.hz
        lyx, V0 = g["lyx0"] + g["lyx1"], self.f["uy"]
        wall = jf / hxf * (lyx + g["lxy"])
        dT = (T[..., 1:] - T[..., :-1]) / hxf
        heat = jf / hxf * dT
        inj = [self.nu * float((V0[..., -1] * wall[..., -1] - V0[..., 0] * wall[..., 0]).sum()),
               self.kappa * float((T[..., -1] * heat[..., -1] - T[..., 0] * heat[..., 0]).sum())]
        lyy = g["lyy0"] + g["lyy1"]
        centre = 2 * (g["lxx"] ** 2 + lyy ** 2 + g["lzz"] ** 2) + (g["lzy"] + g["lyz"]) ** 2
        face = (lyx + g["lxy"]) ** 2 + (g["lzx"] + g["lxz"]) ** 2
        t = T[..., 1:-1]
        dc = ((t - _ym(t)) / self.hyc[1:-1]) ** 2 + ((t - _zm(t)) / hz) ** 2
        dis = [self.nu * float((jc * centre).sum() + (jf * face).sum()), self.kappa * float((jf * dT ** 2).sum() + (jc * dc).sum())]
        U, V, W = (self.f[n] for n in VELOCITY)
        en = [0.5 * float((jf[1:-1] * U[..., 1:-1] ** 2).sum())] + [0.5 * float((jc * q[..., 1:-1] ** 2).sum()) for q in (V, W, T)]
        if not self.kw["scalar"]:   # the library's diagnostics leave out a scalar it does not advance
            inj[1] = dis[1] = en[3] = 0.0
        adv = 0.5 * (_ym(U) + U) * 0.5 * (V[..., :-1] + V[..., 1:])
        st = dict(ux1=U, ux2=U * U, uy1=V, uy2=V * V, uz1=W, uz2=W * W, adv=adv, dif=lyx + g["lxy"])
        return dict(injection=np.array(inj), dissipation=np.array(dis), energy=np.array(en),
                    stats={n: a.cpu().numpy() for n, a in st.items()})


def _network(x, layers):
    """the closure network on x (batch, z, y, x, channel)"""
    for l, (w, b) in enumerate(layers):
        pad = torch.nn.functional.pad(x, (0, 0, 1, 1))
        nx, acc = x.shape[3], b
        for tap in range(27):
            dx, dy, dz = tap % 3 - 1, tap // 3 % 3 - 1, tap // 9 - 1
            shifted = torch.roll(pad[:, :, :, 1 + dx:1 + dx + nx], (-dz, -dy), (1, 2))
            acc = acc + shifted @ w[tap].t()
        x = torch.relu(acc) if l < 2 else acc
    return x


def _exact_layers(seed):
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=_device())  # noqa: E731
    out = []
    for l, (w, b) in enumerate(_layers(seed)):
        out.append((t(w[:, :, :5] if l == 0 else w), t(b)))
    return out


def _exact_train(case, seed):
    x, y = _batch(case, seed)
    x, y = (torch.tensor(a, dtype=torch.float64, device=_device()) for a in (x, y))
    layers = [(w.requires_grad_(), b.requires_grad_()) for w, b in _exact_layers(seed)]
    loss = ((_network(x, layers)[..., :4] - y) ** 2).mean()
    loss.backward()
    out = []
    for l, (w, b) in enumerate(layers):
        row = []
        for p in (w, b):
            row.append((p - 1e-3 * p.grad / (p.grad.abs() + 1e-8)).detach())
        row += [w.grad, b.grad]
        if l == 0:   # the device's rows hold 16 input channels
            row = [torch.nn.functional.pad(a, (0, 11)) if a.dim() == 3 else a for a in row]
        out.append(tuple(a.cpu().numpy() for a in row))
    return {"loss": float(loss), "layers": out}


def _exact_closure(case, seed):
    flow = _Flow(_closure_case(case), _fields(_closure_case(case), seed))
    layers = _exact_layers(seed)
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=_device())  # noqa: E731
    mean, std, scale = (t(a) for a in _closure_norm())
    _, xc, _ = _setup(_closure_case(case))
    r = t(xc[1:-1])
    for _ in range(case["steps"]):
        U, V, W, T = (flow.f[n] for n in ("ux", "uy", "uz", "t"))
        u = 0.5 * (U[..., :-1] + U[..., 1:])
        x = torch.stack([u, V[..., 1:-1], W[..., 1:-1], T[..., 1:-1], r.expand(u.shape)], -1)
        y = _network(((x - mean) / std)[None], layers)[0][..., :4] * scale
        flow.extra = {"ux": 0.5 * (y[..., :-1, 0] + y[..., 1:, 0]), "uy": y[..., 1], "uz": y[..., 2], "t": y[..., 3]}
        dt = flow.step()
    return flow.results(dt)


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "predict":
        x = torch.tensor(_batch(case, seed)[0], dtype=torch.float64, device=_device())
        return _network(x, _exact_layers(seed))[..., :4].cpu().numpy()
    if kind == "closure":
        return _exact_closure(case, seed)
    if kind == "ensemble" or case["nx"] * case["ny"] * case["nz"] > MOST_HOST_CELLS:
        return None
    flow = _Flow(case, _fields(case, seed))
    for _ in range(case["steps"]):
        dt = flow.step()
    out = flow.results(dt)
    if case["logged"]:
        out.update(flow.logged())
    return out
