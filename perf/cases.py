"""Workloads of the library's public entry points, each with its set-up, one
pass, the work the pass cannot do without and, where plain torch in 64 bits
gives it in reasonable time, the result.

A case is a run between two outputs: a simulation (or an ensemble, or a coarse
run with the learned closure) advanced by some steps and its concentration and
velocity read back, as a program does that writes them to a file.  Plain runs
are read as FP64; mixed runs are kept in FP32, the precision of their fields
and of the reference's caf files.
"""
import ctypes
import math

import numpy as np
import torch

import pllcart3d_amd as P
from pllcart3d_amd import closure
from pllcart3d_amd._lib import FIELD_ID

VELO = ("U_OLD", "V_OLD", "W_OLD")

# one substage by the reference's calls (pllcart3d.c:169-194)
SUBSTAGE = ("CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
            "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD")


def _run(name, shape, precision, steps, **kw):
    c = dict(name=name, kind="run", nx=shape[0], ny=shape[1], nz=shape[2], precision=precision, steps=steps,
             R=3.0, Pe=2000.0, thick=0.02, front="modes", Fx=0.0, Fy=0.0, Nmvp=0)
    c.update(kw)
    return c


def listed():
    return [
        # the 64x32x32 reference case watched while it runs: two steps between
        # two looks at the fields, where launches and latency count
        _run("watch_64x32x32", (64, 32, 32), "plain", 2, R=2.0, Pe=500.0, thick=0.05, front="noise"),
        # a test-sized grid with no round number in it, the non-monotonic
        # viscosity law (the reference's shipped param.input setting)
        _run("nmvp_97x45x39", (97, 45, 39), "plain", 20, R=3.0, Pe=300.0, thick=0.1, front="noise", Nmvp=1),
        # gravity (body force) in mixed precision on ragged planes
        _run("gravity_150x70x51_mixed", (150, 70, 51), "mixed", 30, R=2.0, Pe=800.0, thick=0.05, Fx=2.0, Fy=-1.0),
        # planes of the middle range, whose transforms are dense contractions
        _run("front_256x96x96_mixed", (256, 96, 96), "mixed", 30),
        # the 256x128x128 benchmark workload between two outputs
        _run("front_256x128x128", (256, 128, 128), "plain", 30),
        _run("front_256x128x128_mixed", (256, 128, 128), "mixed", 30),
        # the largest configuration
        _run("front_512x256x256", (512, 256, 256), "plain", 12, Pe=4000.0),
        _run("front_512x256x256_mixed", (512, 256, 256), "mixed", 12, Pe=4000.0),
        # a program that calls the operators one by one, one time step
        _run("operators_128x64x64", (128, 64, 64), "plain", 1, kind="operators", Pe=1000.0),
        # a parameter study on the ensemble's three grids
        dict(name="study_24_mixed", kind="ensemble", members=24, shapes="64x32x32 128x48x48 192x64x64",
             precision="mixed", steps=40),
        # the coarse production run with the learned closure and its guard
        _run("closure_128x64x64", (128, 64, 64), "mixed", 20, kind="closure", every=16),
        # training that closure (forward, backward and Adam)
        dict(name="train_64x32x32", kind="train", nx=64, ny=32, nz=32, samples=4, steps=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: grids from 24x12x12 to
    512x256x256, half of them with the square planes of the configurations."""
    kind = rng.choice(["run"] * 7 + ["operators", "ensemble", "closure"])
    if kind == "ensemble":
        sh = [(16 * rng.randint(3, 12), 16 * rng.randint(1, 4), 16 * rng.randint(1, 4)) for _ in range(2)]
        return dict(kind=kind, members=rng.randint(4, 20), shapes=" ".join("x".join(map(str, s)) for s in sh),
                    precision=rng.choice(["mixed", "mixed", "plain"]), steps=2 * rng.randint(2, 15))
    if rng.random() < 0.5:
        ny = nz = rng.choice([32, 48, 64, 96, 128, 128, 256])
        nx = _log(rng, 64, 512)
    else:
        nx, ny = _log(rng, 24, 512), _log(rng, 12, 256)
        nz = min(256, max(12, int(round(ny * 2 ** rng.uniform(-0.7, 0.7)))))
    if kind != "run":
        nx, ny, nz = min(nx, 160), min(ny, 80), min(nz, 80)
    cells = nx * ny * nz
    c = _run("", (nx, ny, nz), rng.choice(["plain", "mixed"]), 2 * max(1, min(20, int(1e8 / cells))), kind=kind,
             R=round(rng.uniform(1.0, 4.0), 3), Pe=float(_log(rng, 200, 4000)), thick=round(rng.uniform(0.03, 0.1), 4),
             front=rng.choice(["modes", "noise"]))
    del c["name"]
    if kind == "run" and rng.random() < 0.25:
        c.update(Fx=round(rng.uniform(-3, 3), 2), Fy=round(rng.uniform(-3, 3), 2))
    if kind == "run" and rng.random() < 0.2:
        # a front that the bisection for the law's slope parameter resolves
        c.update(Nmvp=1, R=round(rng.uniform(2.0, 3.0), 3), nx=max(nx, 48), thick=0.1, front="noise")
    if kind == "operators":
        c.update(steps=1)
    if kind == "closure":
        c.update({n: 8 * max(2, c[n] // 8) for n in ("nx", "ny", "nz")})
        c.update(precision="mixed", steps=20, every=rng.choice([1, 4, 16]))
    return c


# ------------------------------------------------------------------ inputs

def params(c):
    return P.make_params(c["nx"], c["ny"], c["nz"], Vratio=c["R"], Pe=c["Pe"], Inf_thick=c["thick"], Fx=c["Fx"],
                         Fy=c["Fy"], Nmvp=c["Nmvp"])


def front(nx, ny, nz, thick, kind, seed, amp=0.01, dev="cpu"):
    """The initial concentration on every cell, FP64: an erf front at x = 1
    of the box 4x1x1, displaced by 16x16 modes of random phase, or plain with
    noise where 0.01 < c < 0.99."""
    f8 = dict(dtype=torch.float64, device=dev)
    x = (torch.arange(nx + 6, **f8) - 2.5) * (4.0 / nx)
    rng = np.random.default_rng(seed)
    if kind == "modes":
        y = (torch.arange(ny + 2, **f8) - 0.5) / ny
        z = (torch.arange(nz + 2, **f8) - 0.5) / nz
        m = torch.arange(1, 17, **f8)
        ph, ps = (torch.tensor(rng.uniform(0, 2 * math.pi, (16, 16)), **f8) for _ in range(2))
        cy = torch.cos(math.pi * m[:, None, None] * y + ph[:, :, None]).reshape(256, -1)
        cz = torch.cos(math.pi * m[None, :, None] * z + ps[:, :, None]).reshape(256, -1)
        S = cy.t().contiguous() @ cz
        eta = amp * S / S[1:-1, 1:-1].abs().max()
        return 0.5 + 0.5 * torch.erf((x[:, None, None] - 1.0 - eta) / thick)
    c = (0.5 + 0.5 * torch.erf((x - 1.0) / thick))[:, None, None].expand(-1, ny + 2, nz + 2).clone()
    u = torch.tensor(rng.uniform(-1, 1, (nx, ny, nz)), **f8)
    a = c[3:-3, 1:-1, 1:-1]
    a.copy_(torch.where((a > 0.01) & (a < 0.99), (a + amp * u).clamp(0.0, 1.0), a))
    c[3:-3, 0], c[3:-3, -1] = c[3:-3, 1], c[3:-3, -2]
    c[3:-3, :, 0], c[3:-3, :, -1] = c[3:-3, :, 1], c[3:-3, :, -2]
    return c


def _initial(c, seed, dev):
    return front(c["nx"], c["ny"], c["nz"], c["thick"], c["front"], seed, dev=dev)


class Reader:
    """Page-locked host arrays that a simulation's concentration and
    velocity are read into again and again."""

    def __init__(self, sim, precision):
        self.sim = sim
        self.f = [torch.empty((1,) + sim.shape, dtype=torch.float64, pin_memory=True),
                  torch.empty((3,) + sim.shape, dtype=torch.float64, pin_memory=True)]
        self.kept = [torch.empty(a.shape, dtype=torch.float32) for a in self.f] if precision == "mixed" else self.f

    def read(self):
        L, h = self.sim.L, self.sim.h
        for a, names in zip(self.f, (("C_OLD",), VELO)):
            for q, name in enumerate(names):
                if L.pllc_sim_download(h, FIELD_ID[name],
                                       ctypes.cast(a[q].data_ptr(), ctypes.POINTER(ctypes.c_double))) != 0:
                    raise RuntimeError("download: " + P.last_error())
        if self.kept is not self.f:
            for k, a in zip(self.kept, self.f):
                k.copy_(a)
        return {"c": self.kept[0], "velocity": self.kept[1]}


def prepare(c, seed):
    if c["kind"] == "train":
        return _prepare_train(c, seed)
    if c["kind"] == "ensemble":
        rng = np.random.default_rng(seed)
        shapes = [tuple(map(int, s.split("x"))) for s in c["shapes"].split()]
        prm, c0 = [], []
        for m in range(c["members"]):
            sh = shapes[m % len(shapes)]
            prm.append(P.make_params(*sh, Vratio=float(rng.uniform(1, 4)),
                                     Pe=float(np.exp(rng.uniform(np.log(200.0), np.log(4000.0)))), Inf_thick=0.05))
            c0.append(front(*sh, 0.05, "noise", seed * 1000 + m).numpy())
        ens = P.Ensemble(prm, c["precision"])
        for m, a in zip(ens.members, c0):
            m.init(a)
        return dict(case=c, ens=ens, readers=[Reader(m, c["precision"]) for m in ens.members])
    sim = P.Sim(params(c), c["precision"])
    sim.init(_initial(c, seed, "cuda").cpu().numpy())
    s = dict(case=c, sim=sim, reader=Reader(sim, c["precision"]))
    if c["kind"] == "closure":
        net = closure.Network(c["nx"], c["ny"], c["nz"])
        net.set_params(closure.flat_from_dict(closure.init_params(seed)))
        net.set_norm(np.zeros(5), np.ones(5), 1e-3)
        closure.set_closure(sim, net, c["every"])
        s["net"] = net
    return s


def _prepare_train(c, seed):
    """Samples of normalised inputs and targets: smooth in space as filtered
    fields are, of unit size."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = (c["nx"], c["ny"], c["nz"])
    net = closure.Network(*n)
    mask = np.zeros(n, np.uint8)
    mask[closure.XMARGIN:-closure.XMARGIN] = 1
    for _ in range(c["samples"]):
        a = torch.randn((6, 1) + n, generator=g, device="cuda")
        a = torch.nn.functional.avg_pool3d(a, 3, 1, 1, count_include_pad=False)[:, 0]
        a = a / a.std()
        net.add_sample(a[:5].permute(1, 2, 3, 0).contiguous().cpu().numpy(), a[5].contiguous().cpu().numpy(), mask)
    net.set_params(closure.flat_from_dict(closure.init_params(seed)))
    return dict(case=c, net=net, order=np.arange(c["samples"], dtype=np.int32))


# -------------------------------------------------------------------- pass

def run(s):
    c = s["case"]
    if c["kind"] == "train":
        losses = s["net"].train(c["steps"], s["order"], 1e-3)
        return {"losses": losses.astype(np.float32), "weights": s["net"].get_params().astype(np.float32)}
    if c["kind"] == "ensemble":
        s["ens"].run(c["steps"])
        return [r.read() for r in s["readers"]]
    sim = s["sim"]
    if c["kind"] == "closure":
        fallbacks, _ = closure.run_guarded(sim, c["steps"], 10, 2e-2, 1e-4)
        return dict(s["reader"].read(), fallbacks=fallbacks)
    if c["kind"] == "operators":
        dt = min(sim.op("FIND_CFL"), sim.timestep)
        for rk in range(3):
            vbulk = sim.op("BULK_VELO", rk=rk)
            for op in SUBSTAGE:
                sim.op(op, dt, rk, vbulk)
        return dict(s["reader"].read(), dt=dt)
    t, dt = sim.run(c["steps"])
    return dict(s["reader"].read(), t=t, dt=dt)


def work(c):
    """Bytes and operations of one pass.  A substage reads and writes c, u,
    v, w, their explicit terms and the pressure gradient (11 fields) once and
    computes about 2200 operations per cell (four 3-direction WENO terms, the
    twelve line solves, the transforms); the four fields read back cross to
    the host once more."""
    if c["kind"] == "train":
        cells = c["nx"] * c["ny"] * c["nz"]
        conv = 2.0 * 27 * cells * (16 * 5 + 16 * 16 + 16)
        return {"bytes": c["steps"] * cells * (5 + 1 + 4 * 16) * 2.0, "flops": c["steps"] * 3 * conv}
    size = 8 if c["precision"] == "plain" else 4
    if c["kind"] == "ensemble":
        shapes = [tuple(map(int, s.split("x"))) for s in c["shapes"].split()]
        cells = sum(math.prod(shapes[m % len(shapes)]) for m in range(c["members"]))
    else:
        cells = c["nx"] * c["ny"] * c["nz"]
    n = 3 * c["steps"]
    return {"bytes": float(cells * size * (22 * n + 4)), "flops": 2200.0 * cells * n}


# ------------------------------------------------------------ 64-bit result

class Plain64:
    """The time step in plain torch FP64: array expressions for the explicit
    terms, Thomas elimination over whole planes, transforms as matrix
    products.  Fields carry the (3, 1, 1) ghost cells of the library."""

    G, RHO = (8 / 15, 5 / 12, 3 / 4), (0.0, -17 / 60, -5 / 12)

    def __init__(self, c, c0):
        self.c, dev = c, c0.device
        self.n = (c["nx"], c["ny"], c["nz"])
        self.h = (4.0 / c["nx"], 1.0 / c["ny"], 1.0 / c["nz"])
        z = lambda: torch.zeros_like(c0)  # noqa: E731
        self.q = {"c": c0.clone(), "u": z(), "v": z(), "w": z()}
        self.N = {f: z() for f in "cuvw"}
        self.pg = {f: z() for f in "uvw"}
        nx, ny, nz = self.n
        self.lo = {"c": (3, 1, 1), "u": (4, 1, 1), "v": (3, 2, 1), "w": (3, 1, 2)}
        self.hi = (nx + 3, ny + 1, nz + 1)
        y = (torch.arange(ny, dtype=torch.float64, device=dev) + 0.5) / ny - 0.5
        u = self.q["u"]
        u[3, 1:-1, :] = (1.5 * (1 - 4 * y * y))[:, None]
        u[3, 0], u[3, -1] = -u[3, 1], -u[3, -2]
        self.ghosts()
        self.law = self._law(c, c0)
        self.mu = self.viscosity(self.q["c"])
        self.cap = min(2e-3, 0.1 * c["Pe"] * min(self.h) ** 2)
        self.phi, self.t = z(), 0.0
        self.dct, self.lam = [], []
        for n, h in zip(self.n[1:], self.h[1:]):
            k = torch.arange(n, dtype=torch.float64, device=dev)
            self.dct.append(2 * torch.cos(math.pi / n * k[:, None] * (k + 0.5)))
            self.lam.append(2 * (torch.cos(math.pi * k / n) - 1) / h ** 2)

    def _law(self, c, c0):
        M = c["R"]
        if not c["Nmvp"]:
            return lambda a: torch.exp(M * a)
        mum = 1.5 * math.exp(M)
        psi0, psi1 = math.asin(math.exp(M) / mum), math.pi - math.asin(1 / mum)
        etam = (math.pi / 2 - psi0) / (psi1 - psi0)
        shape = lambda cm: ((1 - cm) - etam) / ((1 - cm) * (etam - 1))  # noqa: E731
        # bisection on the centre line: the mean end slope of mu is 0 there
        near = [int(np.argmin(np.abs((np.arange(n) + 0.5) / n - 0.5))) for n in self.n[1:]]
        line = c0[3:-3, 1 + near[0], 1 + near[1]].cpu().numpy()
        first, last = int(np.argmax(line > 1e-5)), int(len(line) - 1 - np.argmax(line[::-1] < 1 - 1e-5))
        first = max(first, 1)
        lo, hi, cm, slope = 0.1, 0.9, 0.5, 1.0
        while abs(slope) > 1e-5:
            a = shape(cm)
            eta = (1 + a) * line / (1 + a * line)
            mu = mum * np.sin(psi0 * (1 - eta) + psi1 * eta)
            slope = ((mu[first + 1] - mu[first]) / (line[first + 1] - line[first]) +
                     (mu[last] - mu[last - 1]) / (line[last] - line[last - 1])) / (math.exp(M) + 1)
            lo, hi = (lo, cm) if slope > 0 else (cm, hi)
            cm = 0.5 * (lo + hi)
        a = shape(cm)

        def law(x):
            eta = (1 + a) * x / (1 + a * x)
            return mum * torch.sin(psi1 * (1 - eta) + psi0 * eta)
        return law

    # a field's unknowns, moved by (i, j, k)
    def at(self, a, f, i=0, j=0, k=0):
        lo, hi = self.lo[f], self.hi
        return a[lo[0] + i:hi[0] + i, lo[1] + j:hi[1] + j, lo[2] + k:hi[2] + k]

    def along(self, a, f, axis, m):
        s = [0, 0, 0]
        s[axis] = m
        return self.at(a, f, *s)

    def ghosts(self):
        q = self.q
        I, J, K = slice(3, -3), slice(1, -1), slice(1, -1)
        for f in "uv":
            q[f][I, J, 0], q[f][I, J, -1] = q[f][I, J, 1], q[f][I, J, -2]
        for f in "uw":
            q[f][I, 0, K], q[f][I, -1, K] = -q[f][I, 1, K], -q[f][I, -2, K]
        for f in "vw":
            q[f][2, J, K] = -q[f][3, J, K]

    def viscosity(self, c):
        e = lambda s, t: 0.25 * (s[0] + s[1] + t[0] + t[1])  # noqa: E731
        m = {k: torch.zeros_like(c) for k in ("cell", "xy", "xz", "yz")}
        m["cell"][2:-2] = self.law(c[2:-2])
        m["xy"][3:-2, 1:, 1:-1] = self.law(e((c[2:-3, :-1], c[3:-2, :-1]), (c[2:-3, 1:], c[3:-2, 1:]))[..., 1:-1])
        m["xz"][3:-2, 1:-1, 1:] = self.law(
            e((c[2:-3, :, :-1], c[3:-2, :, :-1]), (c[2:-3, :, 1:], c[3:-2, :, 1:]))[:, 1:-1])
        m["yz"][3:-3, 1:, 1:] = self.law(
            e((c[3:-3, :-1, :-1], c[3:-3, 1:, :-1]), (c[3:-3, :-1, 1:], c[3:-3, 1:, 1:])))
        return m

    def stale(self, q, f):
        """What the second differences one outside a pass's range hold: those
        an earlier pass left at that index, else 0 (x, y and z passes)."""
        lo, hi, h = self.lo[f], self.hi, self.h
        px, py = q[:, hi[1] - 1, hi[2] - 1].tolist(), q[hi[0] - 1, :, hi[2] - 1].tolist()

        def second(p, axis, m):
            if not lo[axis] <= m < hi[axis]:
                return None
            return ((p[m + 1] - p[m]) / h[axis] - (p[m] - p[m - 1]) / h[axis]) / (2 * h[axis])

        def left(axis, m):
            for p, a in ((py, 1), (px, 0))[2 - axis:]:
                if (v := second(p, a, m)) is not None:
                    return v
            return 0.0
        return [(0.0, 0.0)] + [(left(a, lo[a] - 1), left(a, hi[a])) for a in (1, 2)]

    def upwind(self, q, f, axis, vel, out):
        """ENO2 within two points of a range's ends, WENO5 elsewhere."""
        h, n = self.h[axis], self.hi[axis] - self.lo[f][axis]
        up = vel >= 0
        D = [None] * 6
        for m in range(6):   # the first differences at the faces m-3 .. m+2
            a, b = m - 3, m - 2
            lo, hi = self.lo[f][axis] + a, self.hi[axis] + b
            pad = (max(0, -lo), max(0, hi - q.shape[axis]))
            s = list(zip(self.lo[f], self.hi))
            s[axis] = (max(0, lo), min(q.shape[axis], hi))
            v = q[tuple(slice(*r) for r in s)]
            if any(pad):
                full = [0, 0, 0, 0, 0, 0]
                full[2 * (2 - axis)], full[2 * (2 - axis) + 1] = pad
                v = torch.nn.functional.pad(v, full)
            D[m] = v.diff(dim=axis) / h
        v = [torch.where(up, D[i], D[5 - i]) for i in range(5)]
        c1 = (2 * v[0] - 7 * v[1] + 11 * v[2]) / 6
        c2 = (-v[1] + 5 * v[2] + 2 * v[3]) / 6
        c3 = (2 * v[2] + 5 * v[3] - v[4]) / 6
        s1 = 13 / 12 * (v[0] - 2 * v[1] + v[2]) ** 2 + (v[0] - 4 * v[1] + 3 * v[2]) ** 2 / 4
        s2 = 13 / 12 * (v[1] - 2 * v[2] + v[3]) ** 2 + (v[1] - v[3]) ** 2 / 4
        s3 = 13 / 12 * (v[2] - 2 * v[3] + v[4]) ** 2 + (3 * v[2] - 4 * v[3] + v[4]) ** 2 / 4
        eps = 1e-6 * torch.stack(v).square().amax(0) + 1e-99
        a1, a2, a3 = 0.1 / (s1 + eps) ** 2, 0.6 / (s2 + eps) ** 2, 0.3 / (s3 + eps) ** 2
        w = (a1 * c1 + a2 * c2 + a3 * c3) / (a1 + a2 + a3)
        # second differences at m-1, m, m+1; those outside the range from `out`
        E = [(D[i + 1] - D[i]) / (2 * h) for i in (1, 2, 3)]
        E[0].narrow(axis, 0, 1).fill_(out[0])
        E[2].narrow(axis, n - 1, 1).fill_(out[1])
        d1 = torch.where(up, D[2], D[3])
        a, b = torch.where(up, E[0], E[1]), torch.where(up, E[1], E[2])
        e = d1 + torch.where(a.abs() <= b.abs(), a, b) * h * torch.where(up, 1.0, -1.0)
        m = torch.arange(n, device=q.device)
        end = ((m <= 1) | (m >= n - 2)).reshape([-1 if d == axis else 1 for d in range(3)])
        return torch.where(end, e, w)

    def coefficients(self, f, axis, mu):
        """(a, c) of the diffusion operator's rows; b = -(a + c)."""
        h = self.h[axis]
        if f == "c":
            k = 1 / (self.c["Pe"] * h * h)
            return k, k
        own = "uvw".index(f)
        if axis == own:
            return tuple(2 / (h * h) * self.along(mu["cell"], f, axis, m) for m in (-1, 0))
        e = mu["".join(sorted("xyz"[axis] + "xyz"[own]))]
        return tuple(1 / (h * h) * self.along(e, f, axis, m) for m in (0, 1))

    @staticmethod
    def thomas(a, b, c, r):
        """Lines along the first axis, solved in r."""
        n = r.shape[0]
        cp = torch.empty_like(r)
        den = b[0]
        cp[0] = c[0] / den
        r[0] /= den
        for i in range(1, n):
            den = torch.addcmul(b[i], cp[i - 1], a[i], value=-1)
            torch.div(c[i], den, out=cp[i])
            r[i].addcmul_(r[i - 1], a[i], value=-1).div_(den)
        for i in range(n - 2, -1, -1):
            r[i].addcmul_(cp[i], r[i + 1], value=-1)
        return r

    # the rows next to a wall: +1 Neumann, -1 Dirichlet, 0 a known value
    ENDS = {"c": ((0, 0), (1, 1), (1, 1)), "u": ((0, 0), (-1, -1), (1, 1)), "v": ((-1, 0), (0, 0), (1, 1)),
            "w": ((-1, 0), (-1, -1), (0, 0))}

    def implicit(self, f, S, mu, fac, dt, g, r, vbulk, new):
        old, N, hi = self.q[f], self.N[f], self.hi
        i0 = hi[0]
        face = (slice(i0, i0 + 1),) + tuple(slice(a, b) for a, b in zip(self.lo[f][1:], hi[1:]))
        inner = (slice(i0 - 1, i0),) + face[1:]
        nb = -vbulk * (old[face] - old[inner]) / self.h[0]
        out = dt * (g * nb + r * N[face])
        for axis in (1, 2, 0):
            a, c = self.coefficients(f, axis, mu)
            a, c = (torch.full_like(S, -fac * v) if f == "c" else -fac * v for v in (a, c))
            a, c, S = (x.movedim(axis, 0).contiguous() for x in (a, c, S))
            b = 1 - a - c
            e = self.ENDS[f][axis]
            b[0] += e[0] * a[0]
            b[-1] += e[1] * c[-1]
            if axis == 0:
                S[-1] -= c[-1] * out[0]
            S = self.thomas(a, b, c, S).movedim(0, axis)
        new[f] = old.clone()
        self.at(new[f], f).add_(S)
        new[f][face] += out
        return face, nb

    def explicit(self, f, dt, g, r, cnew):
        q, mu, h, own = self.q, self.mu, self.h, "cuvw".index(f) - 1
        p = q[f]
        A = lambda x, *s: self.at(x, f, *s)  # noqa: E731
        out = self.stale(p, f)
        conv, diff = 0, 0
        for axis in range(3):
            o = q["uvw"[axis]]
            s1 = [0, 0, 0]
            s1[axis] = 1
            if f == "c":
                vel = 0.5 * (A(o) + A(o, *s1))
            elif axis == own:
                vel = A(o)
            else:
                s0 = [0, 0, 0]
                s0[own] = -1
                vel = 0.25 * (A(o) + A(o, *s1) + A(o, *s0) + A(o, *[x + y for x, y in zip(s0, s1)]))
            conv = conv + vel * self.upwind(p, f, axis, vel, out[axis])
            a, c = self.coefficients(f, axis, mu)
            x0, xm, xp = A(p), self.along(p, f, axis, -1), self.along(p, f, axis, 1)
            diff = diff + (a * xm - (a + c) * x0 + c * xp)
        N = -conv
        if f != "c":
            back = [0, 0, 0]
            back[own] = -1
            for axis in range(3):
                if axis == own:
                    continue
                e = mu["".join(sorted("xyz"[axis] + "xyz"[own]))]
                o = q["uvw"[axis]]
                for m, sign in ((1, 1), (0, -1)):
                    s = [0, 0, 0]
                    s[axis] = m
                    N = N + sign / (h[axis] * h[own]) * A(e, *s) * (A(o, *s) - A(o, *[x + y for x, y in zip(s, back)]))
        al = g + r
        S = g * N + r * A(self.N[f]) + al * diff
        if f != "c":
            S = S - al * A(self.pg[f])
            force = {"u": self.c["Fx"], "v": self.c["Fy"]}.get(f, 0.0)
            if force:
                S = S - al * force * 0.5 * (A(cnew) + A(cnew, *back))
        return N, dt * S

    def project(self, new, mu, dt, al):
        u, v, w = (new[f] for f in "uvw")
        I, J, K = slice(3, -3), slice(1, -1), slice(1, -1)
        div = ((u[4:-2, J, K] - u[I, J, K]) / self.h[0] + (v[I, 2:, K] - v[I, J, K]) / self.h[1] +
               (w[I, J, 2:] - w[I, J, K]) / self.h[2]) / (dt * al)
        nx, ny, nz = self.n
        Cy, Cz = self.dct
        X = (div.reshape(-1, nz) @ Cz.t().contiguous()).reshape(nx, ny, nz).permute(1, 0, 2).reshape(ny, -1)
        X = (Cy.contiguous() @ X.contiguous()).reshape(ny, nx, nz).permute(1, 0, 2).contiguous()
        d = 1 / self.h[0] ** 2
        a = torch.full_like(X, d)
        b = (-2 * d + self.lam[0][:, None] + self.lam[1]).expand_as(X).clone()
        mean = b[-1, 0, 0].clone()
        b[0] += d
        b[-1] += d
        b[-1, 0, 0] = mean
        X = self.thomas(a, b, a, X)
        iy, iz = ((C.t() / n * 0.5).contiguous() for C, n in zip(self.dct, (ny, nz)))
        iy[:, 0], iz[:, 0] = 1.0 / (2 * ny), 1.0 / (2 * nz)
        X = (X.reshape(-1, nz) @ iz.t().contiguous()).reshape(nx, ny, nz).permute(1, 0, 2).reshape(ny, -1)
        X = (iy @ X.contiguous()).reshape(ny, nx, nz).permute(1, 0, 2)
        phi = self.phi
        phi[I, J, K] = X
        phi[2, J, K], phi[-3, J, K] = phi[3, J, K], phi[-4, J, K]
        phi[I, 0, K], phi[I, -1, K] = phi[I, 1, K], phi[I, -2, K]
        phi[I, J, 0], phi[I, J, -1] = phi[I, J, 1], phi[I, J, -2]
        for f in "uvw":
            own = "uvw".index(f)
            grad = torch.zeros_like(phi)
            s = [slice(None)] * 3
            s[own] = slice(1, None)
            grad[tuple(s)] = phi.diff(dim=own) / self.h[own]
            G = lambda *m: self.at(grad, f, *m)  # noqa: E731
            self.at(new[f], f).sub_(dt * al * G())
            visc = 0
            for axis in range(3):
                a, c = self.coefficients(f, axis, mu)
                visc = visc + a * self.along(grad, f, axis, -1) - (a + c) * G() + c * self.along(grad, f, axis, 1)
            self.at(self.pg[f], f).add_(G() - 0.5 * dt * al * visc)
        trap = lambda p: float(torch.trapezoid(torch.trapezoid(p[J, K], dx=self.h[2]), dx=self.h[1]))  # noqa: E731
        new["u"][-3, J, K] += trap(new["u"][3]) - trap(new["u"][-3])

    def step(self):
        q, h = self.q, self.h
        I, J, K = slice(3, -3), slice(1, -1), slice(1, -1)
        speed = (0.5 * (q["u"][I, J, K] + q["u"][4:-2, J, K]).abs() / h[0] +
                 0.5 * (q["v"][I, J, K] + q["v"][I, 2:, K]).abs() / h[1] +
                 0.5 * (q["w"][I, J, K] + q["w"][I, J, 2:]).abs() / h[2])
        dt = min(0.3 / float(speed.max()), self.cap)
        for g, r in zip(self.G, self.RHO):
            q = self.q
            al, fac = g + r, 0.5 * dt * (g + r)
            end = q["u"][-4, J, K].reshape(-1)
            vbulk = float(end[int(end.abs().argmax())])
            new, terms = {}, {}

            def update(f, cnew, mu):
                N, S = self.explicit(f, dt, g, r, cnew)
                face, nb = self.implicit(f, S, mu, fac, dt, g, r, vbulk, new)
                terms[f] = (N, face, nb)

            update("c", None, None)
            c = new["c"]
            c[I, 0], c[I, -1] = c[I, 1], c[I, -2]
            c[I, :, 0], c[I, :, -1] = c[I, :, 1], c[I, :, -2]
            mu = self.viscosity(c)
            for f in "uvw":
                update(f, c, mu)
            self.q = new
            self.ghosts()
            self.project(new, mu, dt, al)
            self.ghosts()
            for f, (N, face, nb) in terms.items():
                self.at(self.N[f], f).copy_(N)
                self.N[f][face] = nb
            self.mu = mu
            self.t += al * dt
        self.dt = dt


def exact(c, seed):
    """The run in 64 bits; None for ensembles, the closure's runs and
    training (their networks compute in BF16) and where it takes too long."""
    if c["kind"] not in ("run", "operators"):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rows = 2 * c["nx"] + c["ny"] + c["nz"]
    cells = c["nx"] * c["ny"] * c["nz"]
    # a step, measured: launches, the rows of its line solves, its cells
    if c["steps"] * (0.04 + 3.2e-4 * rows + 1.1e-8 * cells) > 15:
        return None
    s = Plain64(c, _initial(c, seed, dev))
    for _ in range(c["steps"]):
        s.step()
    keep = {"c": s.q["c"][None], "velocity": torch.stack([s.q[f] for f in "uvw"])}
    keep = {k: (v if c["precision"] == "plain" else v.float()).cpu() for k, v in keep.items()}
    return dict(keep, dt=s.dt) if c["kind"] == "operators" else dict(keep, t=s.t, dt=s.dt)
