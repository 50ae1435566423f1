"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is a flow problem of a given size and form.  prepare() makes what a solver has in hand before it
advances the flow: the handle with its metric, and the state in host arrays, uploaded.  run() is one pass of
the caller's loop: a few time steps on the device, then the state back in the caller's arrays.  exact() is
the same discretisation written out in plain torch, in 64 bits: the metric from the coordinates, periodic
ghosts and the inflow and outflow writers, characteristic WENO5 / WENO9 fluxes, central viscous fluxes,
SSP-RK3 / RK4 and the CFL step.

Kinds:
  box, plane   a periodic block (3D / 2D) of decaying turbulence that a simulation carries on from pass to pass
  shock        a solve request: the initial state is uploaded, advanced and fetched (normal shock meeting
               vortices, supersonic inflow and Riemann outflow in x)
  batch        many small independent cases advanced together
"""
import ctypes
import math

import numpy as np
import torch

from shock_amd import shockx

GAMMA, PRANDTL, T0 = 1.4, 0.72, 300.0
CFL = 0.4


# ---- the cases -------------------------------------------------------------------------------------------
def _case(name, kind, n, S, order=4, form="fp64", metric="diag", viscous=True, step="cfl", steps=4, mach=0.5,
          reynolds=2000.0):
    c = {"kind": kind, "n0": n[0], "n1": n[1], "n2": n[2], "S": S, "order": order, "form": form, "metric": metric,
         "viscous": viscous, "step": step, "steps": steps, "mach": mach, "reynolds": reynolds}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest run: a plane periodic block as used for checks against a CPU run; launches decide
        _case("plane-64", "plane", (64, 64, 1), 5, steps=5, reynolds=1000.0),
        # a plane run in ninth order on an odd-sized curvilinear grid, fixed time step
        _case("plane-w9-odd", "plane", (211, 157, 1), 9, step="fixed", steps=5),
        # a large plane run with the three-stage scheme
        _case("plane-large", "plane", (1000, 768, 1), 5, order=3, steps=5),
        # a small request of the solve server
        _case("cube-48", "box", (48, 48, 48), 5, step="fixed", steps=5),
        # a middle-sized ninth-order request, sizes that no tile divides
        _case("box-w9", "box", (97, 85, 106), 9, step="fixed", steps=3),
        # the full metric of a curvilinear grid (verification runs: nine entries instead of three)
        _case("box-full-metric", "box", (119, 96, 104), 5, metric="full", steps=3),
        # inviscid flow, three-stage scheme
        _case("box-inviscid", "box", (128, 128, 144), 5, order=3, viscous=False, steps=4),
        # the headline block, in 64 bits and in the mixed form
        _case("cube-256", "box", (256, 256, 256), 5, steps=8),
        _case("cube-256-mixed", "box", (256, 256, 256), 5, form="mixed", steps=8),
        # shock requests in ninth order, as the shock workload runs them, in both forms
        _case("shock-w9", "shock", (176, 128, 136), 9, step="fixed", steps=4, mach=3.0, reynolds=5000.0),
        _case("shock-w9-mixed", "shock", (144, 112, 128), 9, form="mixed", step="fixed", steps=4, mach=2.5,
              reynolds=5000.0),
        # many small cases at once: planes and boxes of both orders
        _case("batch-small", "batch", (12, 16, 40), 0, step="fixed", steps=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over their logarithm, odd ones among them, every form that the kinds take."""
    kind = rng.choice(["plane", "plane", "box", "box", "box", "shock", "batch"])
    form = rng.choice(["fp64", "fp64", "mixed"])
    S = rng.choice([5, 5, 9])
    order = rng.choice([4, 4, 3])
    step = rng.choice(["cfl", "fixed"])
    reynolds = round(math.exp(rng.uniform(math.log(500.0), math.log(5000.0))), 1)
    if kind == "plane":
        return _case(None, kind, (_log(rng, 24, 900), _log(rng, 24, 900), 1), S, order, form, "full", True, step,
                     rng.choice([3, 4, 5]), reynolds=reynolds)
    if kind == "batch":
        return _case(None, kind, (rng.randint(4, 12), rng.randint(12, 18), rng.randint(24, 44)), 0, 4, form, step="fixed",
                     steps=rng.choice([3, 4, 5]), reynolds=reynolds)
    if kind == "shock":
        return _case(None, kind, tuple(_log(rng, 40, 150) for _ in range(3)), rng.choice([5, 9, 9]), order, form,
                     step="fixed", steps=rng.choice([2, 3, 4]), mach=round(rng.uniform(1.5, 3.0), 2), reynolds=reynolds)
    return _case(None, kind, tuple(_log(rng, 20, 180) for _ in range(3)), S, order, form,
                 rng.choice(["diag", "diag", "full"]), rng.random() < 0.8, step, rng.choice([2, 3, 4]),
                 reynolds=reynolds)


def _members(case, seed):
    """The cases that a batch holds: planes and boxes, both orders, sizes between the two given ones."""
    g = np.random.default_rng(1000 + seed)
    lo, hi = case["n1"], case["n2"]
    out = []
    for k in range(case["n0"]):
        # sizes follow from the case alone, states from the seed
        r = np.random.default_rng([case["n0"], lo, hi, k])
        three = k % 3 != 0
        n = [int(r.integers(lo, hi + 1)) for _ in range(3)]
        m = _case(None, "box" if three else "plane", (n[0], n[1], n[2] if three else 1), 9 if k % 4 == 3 else 5, 4,
                  case["form"], "diag", True, "fixed", case["steps"], 0.5, case["reynolds"])
        out.append((m, int(g.integers(1, 2 ** 31 - 1))))
    return out


# ---- inputs ----------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dims(case):
    return 2 if case["kind"] == "plane" else 3


def _n(case):
    return [case["n0"], case["n1"], case["n2"]]


def _coords(case):
    """Extended coordinates (ghost layers and one more on each side) of a smoothly distorted unit box."""
    d, S, n = _dims(case), case["S"], _n(case)
    g, dev, tp = (S + 1) // 2, _device(), 2.0 * math.pi
    ax = []
    for q in range(3):
        if q >= d:
            ax.append(torch.zeros(1, dtype=torch.float64, device=dev))
            continue
        closed = case["kind"] == "shock" and q == 0
        ax.append(torch.arange(-g - 1, n[q] + g + 1, dtype=torch.float64, device=dev) / (n[q] - 1 if closed else n[q]))
    X, Y, Z = torch.meshgrid(*ax, indexing="ij")
    if d == 2:
        s = 0.02 * torch.sin(tp * X) * torch.sin(tp * Y)
        return X + s, Y - s, torch.zeros_like(X)
    s = torch.sin(tp * X) * torch.sin(tp * Y) * torch.sin(tp * Z)
    if case["kind"] == "shock":
        return X + 0.3 / n[0] * s, Y + 0.2 / n[1] * s, Z - 0.2 / n[2] * s
    if case["metric"] == "full":
        return X + 0.03 * s, Y - 0.02 * s, Z + 0.02 * s
    return X + 0.05 * s, Y, Z


def _random_fields(n, d, gen, count):
    """Periodic random-phase fields of rms one with the energy spectrum k^4 exp(-2 (k/kp)^2)."""
    dev = _device()
    k = [torch.fft.fftfreq(n[q], d=1.0 / n[q], dtype=torch.float64, device=dev) for q in range(d)]
    kk = sum(a * a for a in torch.meshgrid(*k, indexing="ij"))
    kp = min(4.0, min(n[:d]) / 6.0)
    amp = kk.clamp_min(1e-30) ** (0.5 * (5 - d)) * torch.exp(-kk / (kp * kp))
    amp[(0,) * d] = 0.0
    hats = []
    for _ in range(count):
        ph = torch.rand(*n[:d], generator=gen, dtype=torch.float64, device=dev) * (2.0 * math.pi)
        hats.append(torch.polar(amp, ph))
    return k, kk, hats


def _real(h):
    f = torch.fft.ifftn(h).real
    return f / f.square().mean().sqrt()


def _state(case, seed):
    """rho, u, v, w, e on the padded grid (ghosts of periodic faces at rest: the first stage fills them)."""
    d, S, n, mach = _dims(case), case["S"], _n(case), case["mach"]
    g, dev = (S + 1) // 2, _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed) & 0x7FFFFFFF)
    k, kk, hats = _random_fields(n, d, gen, d + 2)
    K = torch.meshgrid(*k, indexing="ij")
    dot = sum(K[q] * hats[q] for q in range(d)) / kk.clamp_min(1e-30)
    vel = [torch.fft.ifftn(hats[q] - K[q] * dot).real for q in range(d)]
    rms = sum(v.square().mean() for v in vel).sqrt()
    shape = tuple(n[q] + S + 1 if q < d else 1 for q in range(3))
    sl = tuple(slice(g, g + n[q]) if q < d else slice(0, 1) for q in range(3))
    ups = 1.0 / (GAMMA * mach * mach)
    full = lambda v: torch.full(shape, float(v), dtype=torch.float64, device=dev)  # noqa: E731
    rho, u, v, w, p = full(1), full(0), full(0), full(0), full(1)
    view = lambda f: f.reshape(tuple(n[q] if q < d else 1 for q in range(3)))  # noqa: E731
    if case["kind"] == "shock":
        m2 = mach * mach
        r = (GAMMA + 1.0) * m2 / ((GAMMA - 1.0) * m2 + 2.0)
        pr = 1.0 + 2.0 * GAMMA / (GAMMA + 1.0) * (m2 - 1.0)
        x = torch.arange(-g, n[0] + g, device=dev) / (n[0] - 1)
        post = (x > 0.3).reshape(-1, 1, 1).expand(shape)
        rho[post], p[post] = r, pr
        u.fill_(1.0)
        u[post] = 1.0 / r
        scale = 0.1
    else:
        rho[sl] += 0.05 * view(_real(hats[d]))
        p[sl] += 0.05 * view(_real(hats[d + 1]))
        scale = 0.5 / mach
    for f, h in zip((u, v, w), vel):
        f[sl] += view(h) * (scale / rms)
    e = 0.5 * (u * u + v * v + w * w) + ups * p / ((GAMMA - 1.0) * rho)
    return [rho, u, v, w, e]


INFLOW = (1.0, 1.0, 0.0, 0.0, 1.0)


def _open(case, seed):
    """One flow problem on the device: handle, metric, uploaded state; the host arrays that the state lives in."""
    shock = case["kind"] == "shock"
    d = _dims(case)
    bc = (shockx.BC_INFLOW_SUPERSONIC, shockx.BC_OUTFLOW_RIEMANN, 0, 0, 0, 0) if shock else (0,) * 6
    h = shockx.Case(dims=d, space_order=case["S"], time_order=case["order"], n=tuple(_n(case)), gamma=GAMMA,
                    mach=case["mach"], reynolds=case["reynolds"], prandtl=PRANDTL, T0=T0, inviscid=not case["viscous"],
                    quirks=0 if case["metric"] == "full" and d == 3 else shockx.QUIRKS_REFERENCE, bc=bc,
                    precision=shockx.MIXED if case["form"] == "mixed" else shockx.FP64, inflow=INFLOW)
    h.build_metric(*[a.cpu().numpy() for a in _coords(case)])
    prim = [a.cpu().numpy() for a in _state(case, seed)]
    h.upload_state(prim)
    s = {"h": h, "out": [a.copy() for a in prim], "prim": prim, "case": case}
    s["ptr"] = (ctypes.c_void_p * 5)(*[a.ctypes.data for a in s["out"]])
    s["tau"] = h.cfl_dt(CFL)
    return s


def prepare(case, seed):
    if case["kind"] == "batch":
        parts = [_open(m, sd) for m, sd in _members(case, seed)]
        b = shockx.Batch([p["h"] for p in parts], [p["tau"] for p in parts])
        return {"parts": parts, "batch": b, "case": case}
    return _open(case, seed)


def _fetch(s):
    # the C entry point with the caller's own arrays, as a C program calls it
    if shockx.lib().shx_download_state(s["h"].h, s["ptr"]) != 0:
        raise RuntimeError("shx_download_state failed")
    return s["out"]


def run(s):
    case = s["case"]
    k = case["steps"]
    if case["kind"] == "batch":
        s["batch"].run(k)
        s["batch"].synchronize()
        return [_fetch(p) for p in s["parts"]]
    if case["kind"] == "shock":
        s["h"].upload_state(s["prim"])
    if case["step"] == "cfl":
        t = s["h"].run_cfl(CFL, k)
        return {"t": t, "state": _fetch(s)}
    s["h"].run(s["tau"], k)
    return {"state": _fetch(s)}


def work(case):
    """Per stage the state read and written, U_n, the RK accumulator and the metric once each; multiplications and
    additions of the scheme per node: characteristic fluxes of each direction, viscous fluxes, the update."""
    if case["kind"] == "batch":
        parts = [work(m) for m, _ in _members(case, 0)]
        return {q: sum(p[q] for p in parts) for q in ("bytes", "flops")}
    d = _dims(case)
    nodes = 1
    for q in range(d):
        nodes *= _n(case)[q]
    per = 5 + 5 + 5 + (7.5 if case["order"] == 4 else 0) + (4 if d == 3 and case["metric"] == "diag" else 10)
    flops = d * ((900 if case["S"] == 5 else 2600) + (350 if case["viscous"] else 0)) + 60
    stages = case["steps"] * case["order"] * nodes
    return {"bytes": stages * per * 8, "flops": stages * flops}


# ---- the same discretisation in plain torch --------------------------------------------------------------
class _Plain:
    """One block in torch, 64 bits: fields on the ghost-padded grid (i, j, k)."""

    IN5 = [1 / 60, -8 / 60, 37 / 60, 37 / 60, -8 / 60, 1 / 60]
    MI5 = [-1 / 90, 25 / 180, -245 / 180, 245 / 180, -25 / 180, 1 / 90]
    DE5 = [-1 / 60, 3 / 20, -3 / 4, 0.0, 3 / 4, -3 / 20, 1 / 60]
    IN9 = [a / 2520 for a in (2, -23, 127, -473, 1627, 1627, -473, 127, -23, 2)]
    MI9 = [a / 75600 for a in (-24, 351, -2649, 15351, -110649, 110649, -15351, 2649, -351, 24)]
    DE9 = [a / 2520 for a in (-2, 25, -150, 600, -2100, 0, 2100, -600, 150, -25, 2)]
    # Balsara-Shu indicators of ninth order: upper triangles of the quadratic forms, sub-stencil by sub-stencil
    IS9 = [
        [(22658, -208501, 364863, -288007, 86329), (482963, -1704396, 1358458, -411487), (1521393, -2462076, 758823),
         (1020563, -649501), (107918,)],
        [(6908, -60871, 99213, -70237, 18079), (138563, -464976, 337018, -88297), (406293, -611976, 165153),
         (242723, -140251), (22658,)],
        [(6908, -51001, 67923, -38947, 8209), (104963, -299076, 179098, -38947), (231153, -299076, 67923),
         (104963, -51001), (6908,)],
        [(22658, -140251, 165153, -88297, 18079), (242723, -611976, 337018, -70237), (406293, -464976, 99213),
         (138563, -60871), (6908,)],
        [(107918, -649501, 758823, -411487, 86329), (1020563, -2462076, 1358458, -288007), (1521393, -1704396, 364863),
         (482963, -208501), (22658,)],
    ]

    def __init__(self, case):
        self.case, self.d, self.S, self.n = case, _dims(case), case["S"], _n(case)
        self.g = (self.S + 1) // 2
        self.ng = [self.n[q] + self.S + 1 if q < self.d else 1 for q in range(3)]
        self.shock = case["kind"] == "shock"
        self.per = [q < self.d and not (self.shock and q == 0) for q in range(3)]
        self.ups = 1.0 / (GAMMA * (case["mach"] * case["mach"]))
        self.suth = 100.4 / T0
        self.psi = 1.0 / case["reynolds"]
        self.heat = 1.0 / ((GAMMA - 1.0) * case["mach"] ** 2 * case["reynolds"] * PRANDTL)
        self.eps = 10.0 * math.sqrt(np.finfo(np.float64).tiny)
        self.quirk = not (case["metric"] == "full")
        self.inn = tuple(slice(self.g, self.g + self.n[q]) if q < self.d else slice(0, 1) for q in range(3))
        self._metric()

    def sh(self, f, dir, off, extra=0):
        """f on the interior in the transverse directions, shifted by off along dir; extra: nodes more at the low end."""
        sl = list(self.inn)
        sl[dir] = slice(self.g + off - extra, self.g + self.n[dir] + off)
        return f[tuple(sl)]

    def line(self, f, dir, off):
        """f on every transverse node and the interior along dir, shifted by off."""
        return f.narrow(dir, self.g + off, self.n[dir])

    def wrap(self, f):
        for q in range(self.d):
            if self.per[q]:
                g, n = self.g, self.n[q]
                f.narrow(q, 0, g).copy_(f.narrow(q, n, g))
                f.narrow(q, g + n, g).copy_(f.narrow(q, g, g))
        return f

    def _metric(self):
        X = _coords(self.case)
        def der(f, q):
            if q >= self.d:
                return None
            sl = [slice(1, -1) if a < self.d else slice(0, 1) for a in range(3)]
            lo, hi = list(sl), list(sl)
            lo[q], hi[q] = slice(0, -2), slice(2, None)
            return -0.5 * f[tuple(lo)] + 0.5 * f[tuple(hi)]
        A = [[der(X[c], q) for q in range(3)] for c in range(3)]     # A[c][q] = d x_c / d xi_q
        o, z = torch.ones_like(A[0][0]), torch.zeros_like(A[0][0])
        if self.d == 2:
            A[2][0], A[2][1], A[0][2], A[1][2], A[2][2] = z, z, z, z, o
        elif self.case["metric"] != "full":
            for c in range(3):
                for q in range(3):
                    if c != q:
                        A[c][q] = z
        (xx, xe, xz), (yx, ye, yz), (zx, ze, zz) = A
        J = (xx * ye * zz + xe * yz * zx + xz * yx * ze - xz * ye * zx - xe * yx * zz - xx * yz * ze)
        m = [(ye * zz - yz * ze) / J, (xz * ze - xe * zz) / J, (xe * yz - xz * ye) / J,
             (yz * zx - yx * zz) / J, (xx * zz - xz * zx) / J, (xz * yx - xx * yz) / J,
             (yx * ze - ye * zx) / J, (xe * zx - xx * ze) / J, (xx * ye - xe * yx) / J, J]
        self.met = [self.wrap(a.contiguous()) for a in m]

    def values(self, U):
        rho, u, v, w, e = U
        p = (rho * (GAMMA - 1) / self.ups * (e - 0.5 * (u * u + v * v + w * w))).abs()
        return {"p": p, "T": (p / rho).abs(), "c": torch.sqrt(self.ups * GAMMA * p / rho),
                "mu": (1.0 + self.suth) * (p / rho) ** 1.5 / (p / rho + self.suth)}

    def faces(self, U, V):
        """Supersonic inflow below, Riemann outflow above, along i."""
        g, n, mach = self.g, self.n[0], self.case["mach"]
        rho, u, v, w, p = INFLOW
        for f, val in zip(U, (rho, u, v, w, 0.5 * (u * u + v * v + w * w) + p / rho / (GAMMA - 1.0) * self.ups)):
            f[:g] = val
        V["p"][:g], V["T"][:g] = p, p / rho
        V["c"][:g] = math.sqrt(self.ups * GAMMA * p / rho)
        V["mu"][:g] = (1.0 + self.suth) * (p / rho) ** 1.5 / (p / rho + self.suth)
        for layer in range(g):
            s, t = g + n - 1 - layer, g + n + layer
            cs, us, cinf = V["c"][s], U[1][s], 1.0 / mach
            un = 0.5 * (us + INFLOW[1]) - (cinf - cs) / (GAMMA - 1.0)
            d1 = (0.5 * (cs + cinf) - 0.25 * (GAMMA - 1.0) * (INFLOW[1] - us)) / cs
            r = U[0][s] * d1 ** (2.0 / (GAMMA - 1.0))
            pn = V["p"][s] * d1 ** (2.0 * GAMMA / (GAMMA - 1.0))
            vs, ws = U[2][s].clone(), U[3][s].clone()
            U[0][t], U[1][t], U[2][t], U[3][t] = r, un, vs, ws
            U[4][t] = 0.5 * (un * un + vs * vs + ws * ws) + pn / r / (GAMMA - 1.0) * self.ups
            V["p"][t], V["c"][t] = pn, torch.sqrt(self.ups * GAMMA * pn / r)
            V["T"][t], V["mu"][t] = V["T"][s], V["mu"][s]

    def _phi5(self, d):
        i0 = 13 * (d[0] - d[1]) ** 2 + 3 * (d[0] - 3 * d[1]) ** 2
        i1 = 13 * (d[1] - d[2]) ** 2 + 3 * (d[1] + d[2]) ** 2
        i2 = 13 * (d[2] - d[3]) ** 2 + 3 * (3 * d[2] - d[3]) ** 2
        a = [k / (i + self.eps) ** 2 for k, i in ((1.0, i0), (6.0, i1), (3.0, i2))]
        s = a[0] + a[1] + a[2]
        return a[0] / s * (d[0] - 2 * d[1] + d[2]) / 3 + (a[2] / s - 0.5) * (d[1] - 2 * d[2] + d[3]) / 6

    def _phi9(self, f, d):
        a = []
        for s, (dk, rows) in enumerate(zip((1 / 126, 10 / 63, 10 / 21, 20 / 63, 5 / 126), self.IS9)):
            q = 0
            for r, row in enumerate(rows):
                q = q + f[s + r] * sum(cf * f[s + r + t] for t, cf in enumerate(row))
            a.append(dk / (q + self.eps) ** 2)
        t = a[0] + a[1] + a[2] + a[3] + a[4]
        q = [d[k] - 4 * d[k + 1] + 6 * d[k + 2] - 4 * d[k + 3] + d[k + 4] for k in range(4)]
        return (a[0] / t * q[0] / 5 + a[2] / t * q[1] / 20 + a[3] / t * (3 * q[1] - 2 * q[2]) / 60
                + a[4] / t * (3 * q[1] - 2 * q[2] + 3 * q[3]) / 60 - (39 * q[1] - 14 * q[2] + 3 * q[3]) / 840)

    def weno(self, dir, U, V, Q):
        m = self.met[3 * dir:3 * dir + 3]
        J, S = self.met[9], self.S
        rho, u, v, w, e = U
        th = u * m[0] + v * m[1] + w * m[2]
        r = (S - 1) // 2
        F = [J * (rho * th)] + [J * (rho * th * a + b * V["p"] * self.ups) for a, b in zip((u, v, w), m)]
        F.append(J * (rho * th * (e + V["p"] / rho * self.ups)))
        C = [rho, rho * u, rho * v, rho * w, rho * e]
        mn = torch.sqrt(m[0] ** 2 + m[1] ** 2 + m[2] ** 2)
        spec = th.abs() + V["c"] * mn
        at = lambda f, o: self.sh(f, dir, o, 1)  # noqa: E731  interfaces i+1/2 of nodes g-1 .. g+n-1
        mean = lambda f: 0.5 * (at(f, 0) + at(f, 1))  # noqa: E731
        Jh, ub, vb, wb, rb, cb = mean(J), mean(u), mean(v), mean(w), mean(rho), mean(V["c"])
        nx, ny, nz = (mean(a / mn) for a in m)
        lam = at(spec, -r)
        for s in range(-r + 1, r + 2):
            lam = torch.maximum(lam, at(spec, s))
        lam = lam * Jh
        g1 = GAMMA - 1.0
        q2 = ub * ub + vb * vb + wb * wb
        un = ub * nx + vb * ny + wb * nz
        gc, hm, s2 = g1 / (cb * cb), 1.0 - 0.5 * g1 * q2 / (cb * cb), math.sqrt(2.0)
        ics = 1.0 / (cb * s2)
        h0 = q2 / 2 + cb * cb / g1
        nul = torch.zeros_like(nx)
        L = [[nx * hm - (vb * nz - wb * ny) / rb, gc * ub * nx, gc * vb * nx + nz / rb, gc * wb * nx - ny / rb, -gc * nx],
             [ny * hm - (wb * nx - ub * nz) / rb, gc * ub * ny - nz / rb, gc * vb * ny, gc * wb * ny + nx / rb, -gc * ny],
             [nz * hm - (ub * ny - vb * nx) / rb, gc * ub * nz + ny / rb, gc * vb * nz - nx / rb, gc * wb * nz, -gc * nz]]
        for sg in (1.0, -1.0):
            L.append([ics * (g1 * q2 / 2 - sg * cb * un)] + [(-g1 * a / cb + sg * b) / s2 for a, b in
                                                            ((ub, nx), (vb, ny), (wb, nz))] + [g1 * ics])
        R = [[nx, ny, nz, ics, ics],
             [ub * nx, ub * ny - rb * nz, ub * nz + rb * ny, ics * (ub + nx * cb), ics * (ub - nx * cb)],
             [vb * nx + rb * nz, vb * ny, vb * nz - rb * nx, ics * (vb + ny * cb), ics * (vb - ny * cb)],
             [wb * nx - rb * ny, wb * ny + rb * nx, wb * nz, ics * (wb + nz * cb), ics * (wb - nz * cb)],
             [q2 / 2 * nx + rb * (vb * nz - wb * ny), q2 / 2 * ny + rb * (wb * nx - ub * nz),
              q2 / 2 * nz + rb * (ub * ny - vb * nx), ics * (h0 + cb * un), ics * (h0 - cb * un)]]
        out = [nul.clone() for _ in range(5)]
        for c in range(5):
            a = {s: sum(L[c][q] * at(F[q], s) for q in range(5)) for s in range(-r, r + 2)}
            b = {s: sum(L[c][q] * at(C[q], s) for q in range(5)) for s in range(-r, r + 2)}
            fp = [0.5 * (a[s - r] + lam * b[s - r]) for s in range(S)]
            fm = [0.5 * (a[r + 1 - s] - lam * b[r + 1 - s]) for s in range(S)]
            dp = [fp[s + 1] - fp[s] for s in range(S - 1)]
            dm = [fm[s] - fm[s + 1] for s in range(S - 1)]
            phi = (-self._phi9(fp, dp) + self._phi9(fm, dm)) if S == 9 else (-self._phi5(dp) + self._phi5(dm))
            for q in range(5):
                out[q] += phi * R[q][c]
        for q in range(5):
            f = lambda s: at(F[q], s)  # noqa: E731, B023
            if S == 9:
                t = (533 * (f(1) + f(0)) - 139 * (f(2) + f(-1)) + 29 * (f(3) + f(-2)) - 3 * (f(4) + f(-3))) / 840
            else:
                t = (-(f(-1) + f(2)) + 7 * (f(0) + f(1))) / 12
            o = out[q] + t
            k = self.n[dir]
            Q[q] -= o.narrow(dir, 1, k) - o.narrow(dir, 0, k)

    def _fac(self, dir, m, J):
        """Newtonian stress contracted with the metric rows: [component][velocity][direction], and the heat factor."""
        a = m[3 * dir:3 * dir + 3]
        fac = [[[None] * 3 for _ in range(3)] for _ in range(3)]
        heat = []
        for b in range(3):
            r = m[3 * b:3 * b + 3]
            dot = r[0] * a[0] + r[1] * a[1] + r[2] * a[2]
            for i in range(3):
                for k in range(3):
                    if i == k:
                        fac[i][k][b] = J * (dot + r[i] * a[i] / 3)
                    else:
                        fac[i][k][b] = J * (r[i] * a[k] - 2.0 / 3.0 * r[k] * a[i])
            heat.append(J * dot)
        return fac, heat

    def derivatives(self, U, V):
        co = self.DE5 if self.S == 5 else self.DE9
        G = {}
        for dir in range(self.d):
            for name, f in (("u", U[1]), ("v", U[2]), ("w", U[3]), ("T", V["T"])):
                o = torch.zeros_like(f)
                acc = sum(cf * self.line(f, dir, k - self.g) for k, cf in enumerate(co) if cf)
                self.line(o, dir, 0).copy_(acc)
                G[name, dir] = o
        return G

    def viscous(self, dir, U, V, G, Q):
        mi, it = (self.MI5, self.IN5) if self.S == 5 else (self.MI9, self.IN9)
        d, S, half = self.d, self.S, self.g
        vel = {"u": U[1], "v": U[2], "w": U[3], "T": V["T"]}
        quirk = dir == 2 and self.quirk

        def half_point(f, cf, side):
            if not quirk:
                return sum(c * self.sh(f, dir, k - half + side) for k, c in enumerate(cf))
            # the stencil's offset along k is taken from j, on the flat array
            i = torch.arange(self.g, self.g + self.n[0], device=f.device).reshape(-1, 1)
            j = torch.arange(self.g, self.g + self.n[1], device=f.device).reshape(1, -1)
            base = (i * self.ng[1] + j) * self.ng[2] + j - half + side
            flat = f.reshape(-1)
            return sum(c * flat[base + k] for k, c in enumerate(cf)).unsqueeze(2)

        dd = [{}, {}]
        for side in (0, 1):
            for name in ("u", "v", "w", "T"):
                for b in range(d):
                    dd[side][name, b] = half_point(vel[name], mi, side) if b == dir else half_point(G[name, b], it, side)
        K = []
        for off in (-1, 0, 1):
            fac, heat = self._fac(dir, [self.sh(a, dir, off) for a in self.met[:9]], self.sh(self.met[9], dir, off))
            K.append((fac, heat, self.sh(V["mu"], dir, off)))
        names = ("u", "v", "w")
        f0, mu0 = K[1][0], K[1][2]

        def mixed(side, get):
            lo, hi = K[side], K[side + 1]
            return 0.5 * (lo[2] * get(lo) + hi[2] * get(hi))

        work = prod = 0.0
        for i in range(3):
            acc = 0.0
            for k in range(3):
                for b in range(d):
                    get = lambda x: x[0][i][k][b]  # noqa: E731, B023
                    acc = acc + (dd[1][names[k], b] * mixed(1, get) - dd[0][names[k], b] * mixed(0, get))
                    prod = prod + (self.sh(G[names[i], dir], dir, 0) * self.sh(G[names[k], b], dir, 0) * mu0 * f0[i][k][b])
            if i < d:
                Q[1 + i] += self.psi * acc
            work = work + self.sh(vel[names[i]], dir, 0) * acc
        heat = 0.0
        for b in range(d):
            get = lambda x: x[1][b]  # noqa: E731, B023
            heat = heat + (dd[1]["T", b] * mixed(1, get) - dd[0]["T", b] * mixed(0, get))
        Q[4] += self.heat * heat + self.psi * (work + prod)

    def residual(self, U):
        for f in U:
            self.wrap(f)
        V = self.values(U)
        if self.shock:
            self.faces(U, V)
        Q = [torch.zeros_like(U[0][self.inn]) for _ in range(5)]
        for dir in range(self.d):
            self.weno(dir, U, V, Q)
        if self.case["viscous"]:
            G = self.derivatives(U, V)
            for dir in range(self.d):
                self.viscous(dir, U, V, G, Q)
        return Q

    def step(self, U, tau):
        """One time step; U keeps the ghosts that the last stage filled."""
        i, J = self.inn, self.met[9][self.inn]
        n = [f[i].clone() for f in U]
        if self.case["order"] == 4:
            co = [(1, 0, 0.5, 0, 1), (1, 0, 0.5, 0, 2), (1, 0, 1.0, 0, 2), (1, 0, 1 / 6, 1 / 6, 0)]
        else:
            co = [(1, 0, 1.0, 0, 0), (0.75, 0.25, 0.25, 0, 0), (1 / 3, 2 / 3, 2 / 3, 0, 0)]
        S = [torch.zeros_like(J) for _ in range(5)]
        for a, b, q, f, m in co:
            R = self.residual(U)
            s = [x[i].clone() for x in U]
            S = [x + m * y for x, y in zip(S, R)]
            inc = [tau / J * (q * x + f * y) for x, y in zip(R, S)]
            rho = a * n[0] + b * s[0] + inc[0]
            U[0][i] = rho
            for c in (1, 2, 4) if self.d == 2 else (1, 2, 3, 4):
                U[c][i] = (a * n[c] * n[0] + b * s[c] * s[0] + inc[c]) / rho

    def cfl(self, U):
        V = self.values([f[self.inn] for f in U])
        tot = 0.0
        for q in range(self.d):
            m = [a[self.inn] for a in self.met[3 * q:3 * q + 3]]
            tot = tot + ((U[1][self.inn] * m[0] + U[2][self.inn] * m[1] + U[3][self.inn] * m[2]).abs()
                         + V["c"] * torch.sqrt(m[0] ** 2 + m[1] ** 2 + m[2] ** 2))
        return CFL / float(tot.max())


def exact(case, seed, batched=False):
    if case["kind"] == "batch":
        return [exact(m, sd, True)["state"] for m, sd in _members(case, seed)]
    nodes = case["n0"] * case["n1"] * case["n2"]
    if nodes * case["steps"] * case["order"] > 5e7:
        return None                                   # minutes in plain torch
    with torch.no_grad():
        P, U, t = _Plain(case), _state(case, seed), 0.0
        tau = P.cfl(U)
        for _ in range(case["steps"]):
            if case["step"] == "cfl":
                tau = P.cfl(U)
            at_start = [f.clone() for f in U]
            P.step(U, tau)
            t += tau
        if batched:
            # a batch keeps the state in place: its ghosts are those of the last step's first stage
            for f, f0 in zip(U, at_start):
                P.wrap(f0)[P.inn] = f[P.inn]
            U = at_start
        out = [f.cpu().numpy() for f in U]
    return {"t": t, "state": out} if case["step"] == "cfl" else {"state": out}
