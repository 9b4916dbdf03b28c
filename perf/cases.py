"""The work that this framework's programs have it do, as timed cases.

A program builds a box (or an ensemble of boxes), loads a velocity field and, where it
follows them, tracers, advances a segment of RK3 steps and takes the state back for its
snapshot or restart file; a diagnostics program asks for the statistics of a field.  The
cases are such segments over the box sizes, shapes, forms and precisions in use: from one
32^3 step, where launches and latency are everything, to the 512^3 shear box with a
million tracers and a box with lines of 1024 points.

``listed()`` gives the named cases, ``draw(rng)`` others of the same ranges,
``prepare(case, seed)`` what the program holds before the segment, ``run(state)`` one
segment, ``work(case)`` the bytes and operations it cannot do without and
``exact(case, seed)`` its result from plain 64-bit torch.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "pandora-2.0_amd"))
import pandora_amd as pa  # noqa: E402

# float32 pi widened to double, the constant of the reference's box length
_PI = float(np.float32(np.pi))
_L = 2.0 * _PI

_FORMS = {"iso": (pa.F_ISOTROPIC, pa.NS_BF_ROT), "bfrot": (pa.F_SHEAR_DNS, pa.NS_BF_ROT),
          "rrot": (pa.F_SHEAR_DNS, pa.NS_R_ROT), "conv": (pa.F_SHEAR_DNS, pa.NS_R_CONV)}


def _box(name, nx, ny, nz, form, prec, steps, **kw):
    case = {"name": name, "kind": "run", "nx": nx, "ny": ny, "nz": nz, "form": form, "prec": prec, "steps": steps,
            "tstep": "fixed", "dt": 0.005, "nu": 0.01, "remesh": 250, "u0": 2.0 / 3.0, "kp": 4.0, "tracers": 0,
            "stats": 0, "spherical": False, "forced": False}
    case.update(kw)
    return case


def listed():
    return [
        # the smallest call: a host program that steps a small decaying box itself and reads it every step
        _box("iso32_step_f64", 32, 32, 32, "iso", "f64", 1),
        # 64^3 decaying turbulence with the statistics of every step, as the reference reports them
        _box("iso64_stats_f64", 64, 64, 64, "iso", "f64", 20, stats=1),
        # Rogallo's rotational form through a remesh of the sheared frame (at step 26)
        _box("rrot128_f64", 128, 128, 128, "rrot", "f64", 32, tstep="decide", remesh=25, u0=0.3),
        # the convective form of the sheared equations
        _box("conv96_f64", 96, 96, 96, "conv", "f64", 10, tstep="decide", nu=0.005),
        # a length with a factor five, time step from the Courant number, spherical truncation
        _box("cfl160_f32", 160, 160, 160, "iso", "f32", 12, tstep="cfl", spherical=True),
        # a box whose sides differ, sheared, with tracers
        _box("box120x48x96_f64", 120, 48, 96, "bfrot", "f64", 12, tstep="decide", nu=0.005, tracers=5000),
        # forced isotropic turbulence (Ornstein-Uhlenbeck, |k| <= 2.5) with tracers
        _box("forced128_f32", 128, 128, 128, "iso", "f32", 24, forced=True, dt=0.002, kp=3.0, tracers=16384),
        # the drop-in workload: 256^3 homogeneous shear in FP64 with 262,144 tracers
        _box("shear256_f64", 256, 256, 256, "bfrot", "f64", 20, tstep="decide", nu=0.005, kp=6.0, tracers=262144),
        # the headline workload: 512^3 homogeneous shear, FP32-mixed, 1,048,576 tracers
        _box("shear512_f32", 512, 512, 512, "bfrot", "f32", 50, tstep="decide", nu=0.005, kp=6.0, tracers=1048576),
        # the long lines of the largest boxes (768 and 1024 points)
        _box("channel768x128x1024_f32", 768, 128, 1024, "bfrot", "f32", 12, tstep="decide", nu=0.001, kp=6.0,
             remesh=500),
        # a batched ensemble of small decaying boxes, 16 of each size
        {"name": "ensemble64_f32", "kind": "ensemble", "sizes": "32,48,64,96", "each": 16, "prec": "f32", "steps": 100},
        # every statistics call on one sheared field
        {"name": "stats256_f64", "kind": "stats", "nx": 256, "ny": 256, "nz": 256, "prec": "f64", "st": 0.3,
         "nu": 0.005},
    ]


# even lengths 2^a 3^b 5^c of the boxes in use
_LENGTHS = [24, 32, 36, 40, 48, 60, 64, 72, 80, 96, 100, 108, 120, 128, 144, 160, 180, 192, 200, 240, 256, 288, 300,
            320, 384, 400, 480, 512]


def _near(x):
    return min(_LENGTHS, key=lambda n: abs(math.log(n / x)))


def draw(rng):
    kind = rng.choice(["run"] * 8 + ["ensemble", "stats"])
    prec = rng.choice(["f64", "f32"])
    if kind == "ensemble":
        sizes = sorted(rng.sample([32, 48, 64, 96, 128], rng.randint(2, 4)))
        return {"kind": "ensemble", "sizes": ",".join(map(str, sizes)), "each": rng.randint(3, 16), "prec": prec,
                "steps": rng.randint(10, 60)}
    form = rng.choice(["iso", "iso", "bfrot", "bfrot", "rrot", "conv"])
    n = _near(math.exp(rng.uniform(math.log(24), math.log(200 if form == "conv" else 512))))
    nx = ny = nz = n
    if rng.random() < 0.35:
        nx, ny, nz = (_near(min(512, max(24, n * rng.choice([0.5, 0.75, 1, 1, 1.5])))) for _ in range(3))
    pts = nx * ny * nz
    if kind == "stats":
        return {"kind": "stats", "nx": nx, "ny": ny, "nz": nz, "prec": "f64", "st": round(rng.uniform(-0.5, 0.5), 3),
                "nu": 0.005}
    # a segment costs at most a tenth to a quarter of the 512^3 one's
    most = 512**3 * 10 // (pts * (2 if prec == "f64" else 1) * (2 if form == "conv" else 1))
    case = _box("", nx, ny, nz, form, prec, max(1, min(most, rng.randint(1, 40))), nu=0.005, kp=rng.choice([3.0, 4.0, 6.0]),
                stats=rng.choice([0, 0, 0, 1]), tracers=rng.choice([0, 0, 1]) * max(100, pts // rng.choice([64, 128])),
                spherical=rng.random() < 0.2)
    del case["name"]
    if form == "iso":
        case.update(tstep=rng.choice(["fixed", "fixed", "cfl"]), dt=min(0.005, 0.6 / max(nx, ny, nz)))
    else:
        case.update(tstep="decide", remesh=250)
    if prec == "f32" and case["stats"]:
        case["stats"] = 0  # records are 64-bit sums of the state: returned where the state is 64-bit
    return case


# ---- inputs -----------------------------------------------------------------
def _waves(case, device):
    """Integer wavenumbers of the stored modes, broadcastable over (i, j, k)."""
    out = []
    for axis, n in enumerate((case["nx"], case["ny"], case["nz"])):
        k = n // 3
        w = list(range(k + 1)) + ([] if axis == 0 else list(range(-k, 0)))
        shape = [1, 1, 1]
        shape[axis] = len(w)
        out.append(torch.tensor(w, dtype=torch.float64, device=device).reshape(shape))
    return out


def _field(case, seed, device="cuda"):
    """A solenoidal random field with E(k) ~ k^4 exp(-2 (k/kp)^2), three complex128 arrays
    (NKI, NKJ, NKK), Hermitian on the i = 0 plane, of rms velocity u0."""
    gen = torch.Generator(device=device).manual_seed(int(seed))
    k1, k2, k3 = _waves(case, device)
    kk = k1 * k1 + k2 * k2 + k3 * k3
    kp = case.get("kp", 4.0)
    amp = kk * torch.exp(-kk / (kp * kp)) / torch.sqrt(kk.clamp(min=1.0))
    u = []
    for _ in range(3):
        z = torch.randn(tuple(kk.shape) + (2,), dtype=torch.float64, device=device, generator=gen)
        u.append(torch.view_as_complex(z) * amp)
    div = (k1 * u[0] + k2 * u[1] + k3 * u[2]) / kk.clamp(min=1.0)
    u = [a - k * div for a, k in zip(u, (k1, k2, k3))]
    for a in u:
        p = a[0]
        mirror = torch.roll(torch.flip(p, (0, 1)), (1, 1), (0, 1)).conj()  # (j, k) -> (-j, -k)
        a[0] = 0.5 * (p + mirror)
    e = sum(float(2.0 * a.abs().square().sum() - a[0].abs().square().sum()) for a in u)
    s = case.get("u0", 2.0 / 3.0) * math.sqrt(3.0 / e)
    return [a * s for a in u]


def _positions(case, seed):
    """Tracers released over the inner eight tenths of the box in each direction."""
    rng = np.random.default_rng(int(seed) + 1)
    return (0.1 + 0.8 * rng.random((case["tracers"], 3))) * _L


def _params(case):
    f_type, form = _FORMS[case["form"]]
    kw = dict(nx=case["nx"], ny=case["ny"], nz=case["nz"], f_type=f_type, ns_deformed=form, nu=case["nu"],
              precision=pa.PDR_FP64 if case["prec"] == "f64" else pa.PDR_FP32_MIXED,
              dealiasing=pa.DEALIASING_SPHERICAL if case["spherical"] else pa.DEALIASING_TWOTHIRD)
    if case["tstep"] == "fixed":
        kw.update(rk3_timestep=pa.RK3_TIMESTEP_FIXED, rk3_dt=case["dt"])
    elif case["tstep"] == "cfl":
        kw.update(rk3_timestep=pa.RK3_TIMESTEP_CFL, rk3_cfl=0.5)
    else:
        kw.update(rk3_timestep=pa.RK3_TIMESTEP_DECIDE, remesh_t=case["remesh"])
    if f_type != pa.F_ISOTROPIC:
        kw.update(deform_s=1.0)
    if case["forced"]:
        kw.update(force_tf=0.2, force_kf=2.5, force_sigma=math.sqrt(0.5), force_stop=1000000, force_seed=3)
    return kw


def _member(case, n):
    return _box("", n, n, n, "iso", case["prec"], case["steps"])


def prepare(case, seed):
    if case["kind"] == "ensemble":
        boxes = []
        for m, n in enumerate(int(s) for s in case["sizes"].split(",") for _ in range(case["each"])):
            one = _member(case, n)
            g = pa.Pandora(**_params(one))
            g.set_state(*(a.cpu().numpy() for a in _field(one, 1000 * seed + m)))
            boxes.append(g)
        return {"case": case, "boxes": boxes, "ensemble": pa.Ensemble(boxes), "t": [0.0] * len(boxes), "step": 1}
    if case["kind"] == "stats":
        g = pa.Pandora(nx=case["nx"], ny=case["ny"], nz=case["nz"], f_type=pa.F_SHEAR_DNS, deform_s=1.0, nu=case["nu"],
                       precision=pa.PDR_FP64)
        b, bi = _frame(case["st"])
        g.set_frame(b.T, bi.T)
        g.set_state(*(a.cpu().numpy() for a in _field(case, seed)))
        return {"case": case, "box": g}
    g = pa.Pandora(**_params(case))
    g.set_state(*(a.cpu().numpy() for a in _field(case, seed)))
    if case["tracers"]:
        g.set_particles(_positions(case, seed))
    if case["stats"]:
        g.set_stage_stats(case["stats"])
    return {"case": case, "box": g, "t": 0.0, "step": 1}


# ---- one pass ---------------------------------------------------------------
def _held(case, a):
    """The array as the program keeps it: an FP32-mixed box holds single precision."""
    if case["prec"] == "f64":
        return a
    a = torch.from_numpy(a)
    return a.to(torch.complex64 if a.is_complex() else torch.float32)


def run(state):
    case = state["case"]
    if case["kind"] == "stats":
        g = state["box"]
        spec, q = g.stats()
        rs = g.rs_stats()
        r1i, lint = g.rs_correlation()
        s1, s2, homog = g.spectra_1d()
        return {"spec": np.array(list(spec.values())), "q": np.array(list(q.values())),
                "rs": np.array(list(rs.values())), "r1i": r1i, "lint": lint, "s1": s1, "s2": s2,
                "homog": np.array(list(homog.values()))}
    if case["kind"] == "ensemble":
        state["t"] = state["ensemble"].run(state["step"], case["steps"], state["t"])
        state["step"] += case["steps"]
        out, each = [], case["each"]
        for s in range(len(case["sizes"].split(","))):
            boxes = state["boxes"][s * each:(s + 1) * each]
            snap = [torch.empty((each,) + boxes[0].shape, dtype=torch.complex128 if case["prec"] == "f64" else torch.complex64)
                    for _ in range(3)]
            for m, g in enumerate(boxes):
                for a, b in zip(snap, g.get_state()):
                    a[m].copy_(torch.from_numpy(b))
            out += snap
        return out
    g = state["box"]
    if case["steps"] == 1:
        state["t"] = g.rk3_calc(state["step"], state["t"])
    else:
        state["t"] = g.run(state["step"], case["steps"], state["t"])
    state["step"] += case["steps"]
    out = {"u": [_held(case, a) for a in g.get_state()]}
    if case["tracers"]:
        out["particles"] = [_held(case, a) for a in g.get_particles()]
    if case["stats"]:
        _, q, spec, rs, s1, s2, homog = g.stage_stats()
        out["record"] = {"spec": np.array(list(spec.values())), "q": np.array(list(q.values())),
                         "rs": np.array(list(rs.values())), "s1": s1, "s2": s2,
                         "homog": np.array(list(homog.values()))}
    return out


# ---- what a pass cannot do without ------------------------------------------
def _step_work(case):
    """Bytes and operations of one RK3 step: each stage reads and writes the velocity and the RK
    registers and does nine real 3-D transforms' worth of butterflies and the products."""
    sc = 16 if case["prec"] == "f64" else 8
    pts = case["nx"] * case["ny"] * case["nz"]
    modes = (case["nx"] // 3 + 1) * (2 * (case["ny"] // 3) + 1) * (2 * (case["nz"] // 3) + 1)
    fields = 15 if case["form"] == "conv" else 9
    flops = 3 * (fields * 2.5 * pts * math.log2(pts) + 30.0 * pts + 150.0 * modes)
    moved = 3 * (12 * modes * sc + 96 * case["tracers"])
    return moved, flops + 3 * case["tracers"] * 1000.0, 3 * modes * sc + 48 * case["tracers"]


def work(case):
    if case["kind"] == "stats":
        pts = case["nx"] * case["ny"] * case["nz"]
        modes = (case["nx"] // 3 + 1) * (2 * (case["ny"] // 3) + 1) * (2 * (case["nz"] // 3) + 1)
        return {"bytes": 3 * 16 * modes, "flops": 6 * 2.5 * pts * math.log2(pts) + 60.0 * pts + 100.0 * modes}
    if case["kind"] == "ensemble":
        parts = [_step_work(_member(case, int(n))) for n in case["sizes"].split(",")]
        return {"bytes": case["each"] * sum(p[0] * case["steps"] + p[2] for p in parts),
                "flops": case["each"] * case["steps"] * sum(p[1] for p in parts)}
    moved, flops, kept = _step_work(case)
    return {"bytes": case["steps"] * moved + kept, "flops": case["steps"] * flops}


# ---- the same in plain 64-bit torch -----------------------------------------
def _frame(st):
    """bmat, binv (rows m, columns n) of a frame sheared by st = S t."""
    b, bi = np.eye(3), np.eye(3)
    b[0, 2], bi[0, 2] = -st, st
    return b, bi


class _Plain:
    """The pseudo-spectral RK3 step written with torch.fft."""

    def __init__(self, case, u, x=None):
        self.case, self.u, self.dev = case, u, u[0].device
        self.n = (case["nx"], case["ny"], case["nz"])
        self.k = [k.reshape(k.shape + (1,) * (u[0].dim() - 3)) for k in _waves(case, self.dev)]  # boxes of a batch last
        self.kk = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.at = [torch.cat([torch.arange(n // 3 + 1), torch.arange(n - n // 3, n)]).to(self.dev) for n in self.n[1:]]
        self.form = case.get("form", "bfrot")
        self.rogallo = self.form in ("rrot", "conv")
        self.shear = 0.0 if self.form == "iso" else 1.0
        self.B, self.BI = _frame(0.0)
        self.rk = [torch.zeros_like(a) for a in u]
        self.x = x
        self.up = None if x is None else torch.zeros_like(x)

    def real(self, a):
        nx, ny, nz = self.n
        f = torch.zeros((a.shape[0], ny, nz) + a.shape[3:], dtype=torch.complex128, device=self.dev)
        f[:, self.at[0][:, None], self.at[1]] = a
        f = torch.fft.ifftn(f, dim=(1, 2), norm="forward")
        f[0].imag.zero_()
        return torch.fft.irfft(f, n=nx, dim=0, norm="forward")

    def wave(self, r):
        f = torch.fft.rfft(r, dim=0, norm="forward")[: self.n[0] // 3 + 1]
        f = torch.fft.fftn(f, dim=(1, 2), norm="forward")
        return f[:, self.at[0][:, None], self.at[1]]

    def mix(self, m, v):
        return [sum(float(m[r, c]) * v[c] for c in range(3) if m[r, c] != 0.0) for r in range(3)]

    def kappa(self):  # laboratory wavenumber, sum_m bmat(m, n) k_m
        return self.mix(self.B.T, self.k)

    def mask(self):
        if self.case.get("spherical"):
            kx = self.kappa()
            keep = torch.sqrt(kx[0] ** 2 + kx[1] ** 2 + kx[2] ** 2) <= min(self.n) // 3
            self.u = [a * keep for a in self.u]

    def curl(self, v):
        kx = self.kappa()
        return [1j * (kx[(c + 1) % 3] * v[(c + 2) % 3] - kx[(c + 2) % 3] * v[(c + 1) % 3]) for c in range(3)]

    def nonlinear(self, ur):
        if self.form == "conv":
            w = [sum(float(self.B[d, j]) * ur[j] for j in range(3) if self.B[d, j] != 0.0) for d in range(3)]
            return [self.wave(sum(w[d] * self.real(1j * self.k[d] * a) for d in range(3))) for a in self.u]
        v = ur if self.rogallo else self.mix(self.BI, ur)
        o = [self.real(a) for a in self.curl(self.u if self.rogallo else self.mix(self.BI, self.u))]
        nl = [self.wave(o[(c + 1) % 3] * v[(c + 2) % 3] - o[(c + 2) % 3] * v[(c + 1) % 3]) for c in range(3)]
        return nl if self.rogallo else self.mix(self.B, nl)

    def interpolate(self, ur):
        """Cubic through the 4 x 4 x 4 nodes round every tracer, over the periodic box."""
        at, wt = [], []
        for c, n in enumerate(self.n):
            s = self.x[:, c] / (_L / n)
            first = torch.floor(s).long() - 1
            s = s - first
            node = torch.arange(4, device=self.dev)
            at.append((first[:, None] + node) % n)
            wt.append(torch.stack([math.prod(1.0 / (a - b) for b in range(4) if b != a) * torch.stack(
                [s - b for b in range(4) if b != a]).prod(0) for a in range(4)], 1))
        out = torch.zeros_like(self.x)
        for a in range(4):
            for b in range(4):
                for d in range(4):
                    w = wt[0][:, a] * wt[1][:, b] * wt[2][:, d]
                    for c in range(3):
                        out[:, c] += w * ur[c][at[0][:, a], at[1][:, b], at[2][:, d]]
        return out

    def advance(self, ur, beta, gdt):
        uf = self.interpolate(ur)
        bf = self.form == "bfrot"
        b, bi = (torch.tensor(m, device=self.dev) for m in (self.B, self.BI))
        self.up = beta * self.up + (uf @ bi.T if bf else uf)
        x = (self.x @ bi.T if bf else self.x) + gdt * self.up
        x = x @ b.T if bf else x
        for c, n in enumerate(self.n):
            low = -0.5 * (_L / n)
            x[:, c] += torch.where(x[:, c] < low, _L, 0.0)
            x[:, c] -= torch.where(x[:, c] >= low + _L, _L, 0.0)
        self.x = x

    def update(self, nl, beta, gdt):
        case, k, kx = self.case, self.k, self.kappa()
        p4 = kx[0] ** 2 + kx[1] ** 2 + kx[2] ** 2
        A = np.zeros((3, 3))
        A[0, 2] = self.shear
        H = A if self.rogallo else 2.0 * (self.B @ A @ self.BI)  # the source term's tensor
        kp = kx if self.rogallo else k
        p1 = kx if self.rogallo else self.mix(self.B, kx)
        hu = self.mix(H, self.u)
        push = sum(kp[c] * (nl[c] + hu[c]) for c in range(3)) / p4.clamp(min=1e-300)
        keep = self.kk > 0
        for c in range(3):
            t = -case["nu"] * p4 * self.u[c] - nl[c] + p1[c] * push - hu[c]
            self.rk[c] = torch.where(keep, beta * self.rk[c] + t, self.rk[c])
        u = [torch.where(keep, a + gdt * r, a) for a, r in zip(self.u, self.rk)]
        um = self.mix(self.B, u) if self.rogallo else u
        div = sum(k[c] * um[c] for c in range(3)) / self.kk.clamp(min=1.0)
        um = [a - k[c] * div for c, a in enumerate(um)]
        self.u = self.mix(self.BI, um) if self.rogallo else um

    def remesh(self):
        """The grid sheared by half a box becomes the one sheared by minus half a box: k3 -> k3 - k1."""
        km = self.n[2] // 3
        out = [torch.zeros_like(a) for a in self.u]
        for i in range(self.u[0].shape[0]):
            k = self.k[2].reshape(-1).long()
            new = k - i
            ok = new.abs() <= km
            src = torch.nonzero(ok).reshape(-1)
            dst = new[ok] % (2 * km + 1)
            for a, b in zip(out, self.u):
                a[i][:, dst] = b[i][:, src]
        if not self.rogallo:
            out[0] = out[0] + out[2]
        self.u = out

    def steps(self, first, count, t, before_last=None):
        case = self.case
        for step in range(first, first + count):
            if before_last is not None and step == first + count - 1:
                before_last(self)
            start, dt = t, None
            for beta, gamma, frac in ((0.0, 1 / 3, 1 / 3), (-5 / 9, 15 / 16, 3 / 4), (-153 / 128, 8 / 15, 1.0)):
                if dt is None and self.shear and (step - case["remesh"] - 1) % (2 * case["remesh"]) == 0:
                    assert self.x is None
                    self.remesh()
                    self.B, self.BI = _frame(-0.5)
                self.mask()
                ur = [self.real(a) for a in self.u]
                if dt is None:
                    if case["tstep"] == "fixed":
                        dt = case["dt"]
                    elif case["tstep"] == "cfl":
                        dt = 0.5 * (_L / self.n[0]) / float(sum(a.abs() for a in ur).max())
                    else:
                        dt = 0.5 / case["remesh"]
                nl = self.nonlinear(ur)
                if self.x is not None:
                    self.advance(ur, beta, gamma * dt)
                self.update(nl, beta, gamma * dt)
                self.mask()
                t = start + frac * dt
                if self.shear:
                    late = 0 if step <= case["remesh"] else 1 + (step - case["remesh"] - 1) // (2 * case["remesh"])
                    self.B, self.BI = _frame(t - late)
        return t

    # statistics of the current field
    def statistics(self):
        nu = self.case["nu"]
        kx = self.kappa()
        km = torch.sqrt(kx[0] ** 2 + kx[1] ** 2 + kx[2] ** 2)
        v = self.u if self.rogallo else self.mix(self.BI, self.u)
        two = torch.full((self.u[0].shape[0], 1, 1), 2.0, dtype=torch.float64, device=self.dev)
        two[0] = 1.0
        ph = [two * (v[a].conj() * v[b]).real for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))]
        kkmax = round(math.sqrt(sum((n // 3) ** 2 for n in self.n)))
        e = 0.5 * (ph[0] + ph[1] + ph[2])
        shell = torch.floor(km + 0.5).long().expand(e.shape)
        raw = torch.zeros((7, kkmax), dtype=torch.float64, device=self.dev)
        ok = (shell >= 1) & (shell <= kkmax)
        for q, w in enumerate((e, 0.5 * ph[0], 0.5 * ph[1], 0.5 * ph[2], 2 * nu * km**2 * e, 4 * nu**2 * km**4 * e,
                               two.expand(e.shape))):
            raw[q] = torch.bincount(shell[ok] - 1, weights=w.expand(e.shape)[ok], minlength=kkmax)
        raw = raw.cpu().numpy()
        kk = np.arange(1, kkmax + 1, dtype=float)
        dens = raw[6] / (4.0 / 3.0 * _PI * ((kk + 0.5) ** 3 - (kk - 0.5) ** 3))
        spec = np.zeros((7, kkmax))
        has = dens != 0.0
        spec[:6, has] = raw[:6, has] / dens[has]
        spec[6] = dens
        uu = [float(p.sum()) for p in ph]
        fn = spec[:6].sum(1)
        u1 = math.sqrt(2.0 * fn[0] / 3.0)
        tay = math.sqrt(15.0 * nu * u1 * u1 / fn[4])
        li = [float((_PI / 2.0 / (u1 * u1) * spec[a] / kk).sum()) for a in range(4)]
        q = [0.5 * sum(uu[:3])] + uu + [raw[0, has].sum(), raw[4, has].sum(), raw[5, has].sum()] + list(fn)
        q += [u1] + [math.sqrt(2.0 * fn[a]) for a in (1, 2, 3)]
        q += [fn[0] / fn[4], fn[0] ** 1.5 / fn[4], tay, tay * u1 / nu] + li
        q += [li[0] / u1, (nu**3 / fn[4]) ** 0.25, math.sqrt(nu / fn[4]),
              fn[5] * (15.0 / fn[4]) ** 1.5 * math.sqrt(nu) / 35.0, fn[4] * li[0] / u1**3]
        # the grid's moments: laboratory velocity by binv in every sheared form, the step's vorticity
        ur = [self.real(a) for a in self.u]
        vr = self.mix(self.BI, ur)
        # (in the convective form the record's vorticity slots hold du/dx, the reference's u4..u6)
        om = [self.real(a) for a in ([1j * self.k[0] * b for b in self.u] if self.form == "conv" else self.curl(v))]
        mean = lambda a: float(a.mean())  # noqa: E731
        m2 = [mean(a * a) for a in vr]
        rs = m2 + [mean(vr[0] * vr[1]), mean(vr[0] * vr[2]), mean(vr[1] * vr[2])]
        rs += [mean(a**3) / s**1.5 for a, s in zip(vr, m2)] + [mean(a**4) / s**2 for a, s in zip(vr, m2)]
        rms = [math.sqrt(mean(a * a)) for a in om]
        rms[0] *= math.sqrt(float(np.prod(self.n)))  # the reference leaves this one a sum
        rs += rms + [mean(a**3) / s**3 for a, s in zip(om, rms)] + [mean(a**4) / s**4 for a, s in zip(om, rms)]
        rs += [float(a.abs().max()) for a in om] + [float(sum(a.abs() for a in vr).max())]
        # streamwise spectra (Parseval over y and z) and the homogeneous record
        vl = self.mix(self.BI, self.u)
        f = 2.0 * self.n[1] * self.n[2] / self.n[0] ** 2
        s1, s2 = (f * a.abs().square().sum((1, 2)).cpu().numpy() for a in vl[:2])
        l11 = _PI * s1[0] / (2.0 * uu[0])
        homog = [q[28] * self.shear, 2.0 * uu[0] / (uu[1] + uu[2]), math.inf, *li[1:], l11, 0.0, 0.0, *fn[1:4], *q[17:20]]
        corr = torch.fft.irfft((torch.fft.rfft(vr[0], dim=0).conj() * torch.fft.rfft(ur[0], dim=0)).sum((1, 2)),
                               n=self.n[0]) / float((vr[0] * vr[0]).sum())
        r1i = corr[: self.n[0] // 2 + 1].cpu().numpy()
        return ({"spec": spec, "q": np.array(q), "rs": np.array(rs), "s1": s1, "s2": s2, "homog": np.array(homog)},
                {"r1i": r1i, "lint": float(r1i.sum() * (_L / self.n[0]))})


def exact(case, seed):
    if case["kind"] == "ensemble":
        out, m = [], 0
        for n in (int(s) for s in case["sizes"].split(",")):
            one = _member(case, n)
            fields = [_field(one, 1000 * seed + m + b) for b in range(case["each"])]
            m += case["each"]
            p = _Plain(one, [torch.stack([f[c] for f in fields], -1) for c in range(3)])
            p.steps(1, case["steps"], 0.0)
            out += [a.movedim(-1, 0).contiguous() for a in p.u]
        return out
    if case["kind"] == "stats":
        p = _Plain(case, _field(case, seed))
        p.B, p.BI = _frame(case["st"])
        a, b = p.statistics()
        return {**a, **b}
    if case["forced"]:
        return None  # the forcing's deviates come from the library's own generator
    x = torch.from_numpy(_positions(case, seed)).to("cuda") if case["tracers"] else None
    p = _Plain(case, _field(case, seed), x)
    record = []
    p.steps(1, case["steps"], 0.0, (lambda s: record.append(s.statistics()[0])) if case["stats"] else None)
    out = {"u": p.u}
    if case["tracers"]:
        out["particles"] = [p.x, p.up]
    if case["stats"]:
        out["record"] = record[0]
    return out
