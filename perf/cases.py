"""Performance cases of the MHD time step: what a user of this package runs.

A case is a dict of plain values.  Two kinds of call are measured:

* ``forward`` -- ``Engine.step(steps)`` on a state that lives on the GPU, the
  loop of every simulation; the outputs are the evolved fields, read in place
  (``Engine.device_ptr``).  The run goes on from pass to pass, as a time loop
  does; with ``restart`` each pass starts again from a checkpoint in device
  memory (``Engine.load_pert``, ``Engine.set_clock``), as ensembles and
  parameter studies do.
* ``tangent`` -- ``Engine.tl_step(steps)`` and ``Engine.tl_get()``: the
  forward-mode derivative along the trajectory, whose states and tangents a
  loss function reads on the host.

``exact`` restates the step in float64 torch on whole arrays, without this
package's kernels: the same masks, halo rules and boundary maps, written as
array expressions.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from smaug_amd import configs
from smaug_amd.engine import Engine
from smaug_amd.params import PREC_MIXED, RunParams

GAMMA = 5.0 / 3.0


def _case(name, kind, problem, n, steps, rk=True, mixed=False, driver="vertical", restart=False):
    c = {"kind": kind, "problem": problem, "ndim": len(n), "n0": n[0], "n1": n[1], "n2": n[2] if len(n) == 3 else 1,
         "steps": steps, "rk": rk, "mixed": mixed, "driver": driver, "restart": restart}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # smallest 3D run (the smoke test's grid), a step from a checkpoint:
        # launches and the latency of one tile are all there is
        _case("strat3d_16x12x12", "forward", "stratified", (16, 12, 12), 1, restart=True),
        # 2D Orszag-Tang vortex, periodic, CFL time step, RK4: a short run
        # from a checkpoint
        _case("ot2d_128", "forward", "orszag_tang", (128, 128), 10, driver="none", restart=True),
        # the single-stage scheme on a 2D grid whose sizes fit no tile
        _case("ot2d_250_euler", "forward", "orszag_tang", (250, 250), 10, rk=False, driver="none", restart=True),
        # 2D slice of the stratified atmosphere with the vertical driver
        _case("slice2d_256x512", "forward", "stratified", (256, 512), 5),
        # the same slice with FP32 stencils
        _case("slice2d_256x512_mixed", "forward", "stratified", (256, 512), 5, mixed=True),
        # ragged 3D grid, single-stage scheme, torsional driver, from a checkpoint
        _case("strat3d_101x75x61_euler", "forward", "stratified", (101, 75, 61), 4, rk=False, driver="torsional",
              restart=True),
        # the ordinary 3D run
        _case("strat3d_128", "forward", "stratified", (128, 128, 128), 1),
        # the large 3D run, FP64 and mixed precision
        _case("strat3d_256", "forward", "stratified", (256, 256, 256), 1),
        _case("strat3d_256_mixed", "forward", "stratified", (256, 256, 256), 1, mixed=True),
        # derivative along the slice's trajectory (background direction too)
        _case("tangent2d_256x512", "tangent", "stratified", (256, 512), 10),
        # derivative of a 3D run, FP64 pairs and FP32 pairs
        _case("tangent3d_96", "tangent", "stratified", (96, 96, 96), 10),
        _case("tangent3d_96_mixed", "tangent", "stratified", (96, 96, 96), 10, mixed=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: 2D grids of about 40^2 to 500^2 cells, 3D
    grids of 12^3 to 110^3 (64^3 for tangent runs; the listed 3D runs go on to
    256^3), any aspect within 2:1, each precision, scheme and driver."""
    kind = rng.choice(["forward", "forward", "forward", "tangent"])
    mixed = rng.random() < 0.35
    rk = rng.random() < 0.75

    def around(size, lo):
        return max(lo, int(round(size * rng.uniform(0.75, 1.4))))

    if rng.random() < 0.35:
        size = _log_int(rng, 40, 500)
        n = (around(size, 30), around(size, 30))
        if kind == "forward" and not mixed and rng.random() < 0.4:
            return _case(None, kind, "orszag_tang", n, rng.randint(2, 10), rk, False, "none", True)
        return _case(None, kind, "stratified", n, rng.randint(2, 10), rk, mixed, rng.choice(["vertical", "none"]),
                     kind == "forward" and not rk)
    size = _log_int(rng, 12, 110 if kind != "tangent" else 64)
    n = (around(size, 10), around(size, 10), around(size, 10))
    steps = rng.randint(1, 3) if size > 60 else rng.randint(1, 8)
    driver = rng.choice(["vertical", "torsional", "none"])
    return _case(None, kind, "stratified", n, steps, rk, mixed, driver, kind == "forward" and (not rk or size < 40))


# --------------------------------------------------------------------------
# inputs


def _params(case) -> RunParams:
    n = [case["n0"], case["n1"], case["n2"]][: case["ndim"]]
    if case["problem"] == "orszag_tang":
        rp = configs.orszag_tang_params(ni=n[0], rkon=int(case["rk"]))
        rp.ni = list(n)
    else:
        rp = configs.stratified_params(ni=n, ndim=len(n), rkon=int(case["rk"]))
        if not case["rk"]:
            rp.dt *= 0.2  # the single-stage scheme needs a smaller step
            rp.moddton = 1  # and takes the CFL rule, capped by it
        if case["driver"] == "torsional":
            configs.fluxtube1_driver(rp, centre=(0.6e6, 2.0e6, 2.0e6), widths=(0.3e6, 0.5e6, 0.5e6))
        elif case["driver"] == "none":
            rp.driver = 0
        else:
            # a footprint of a few cells at the bottom, mid-period
            dx = rp.dx
            rp.drv[2:] = [rp.xmin[0] + 2.5 * dx[0], 2.0e6, 2.0e6, 3.0 * dx[0], 3.0 * dx[1]] + [0.0] * 5
            rp.qt0 = 75.0
    if case["mixed"]:
        rp.precision = PREC_MIXED
    return rp


def _axes(rp):
    """Cell-centre coordinates per dim, two ghost cells per side."""
    return [rp.xmin[d] + (np.arange(rp.n[d], dtype=np.float64) - 1.5) * rp.dx[d] for d in range(rp.ndim)]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _smooth(a):
    """Three passes of the periodic 3-point box filter along every axis."""
    for ax in range(a.dim()):
        for _ in range(3):
            a = (a + torch.roll(a, 1, ax) + torch.roll(a, -1, ax)) / 3.0
    return a


def _initial(case, rp, seed):
    """(state, positions): float64 tensors of shapes (nvar, *grid) and
    (ndim, *grid), grid = (n2, n1, n0)."""
    dev, nd = _device(), rp.ndim
    shape = tuple(rp.n[::-1])
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    axes = [torch.tensor(a, device=dev) for a in _axes(rp)]
    pos = torch.stack([axes[d].reshape([-1 if nd - 1 - q == d else 1 for q in range(nd)]).expand(shape)
                       for d in range(nd)])

    def noise(amp):
        return amp * _smooth(torch.randn(shape, generator=gen, device=dev, dtype=torch.float64))

    w = torch.zeros((4 + 3 * nd,) + shape, dtype=torch.float64, device=dev)
    if case["problem"] == "orszag_tang":
        x, y = pos[0], pos[1]
        tp = 2.0 * math.pi
        b0 = 1.0 / math.sqrt(4.0 * math.pi)
        rho = 25.0 / (36.0 * math.pi) * (1.0 + noise(0.05))
        vx, vy = -torch.sin(tp * y) + noise(0.05), torch.sin(tp * x) + noise(0.05)
        bx, by = b0 * (noise(0.05) - torch.sin(tp * y)), b0 * (noise(0.05) + torch.sin(2.0 * tp * x))
        pr = 5.0 / (12.0 * math.pi)
        w[0], w[1], w[2], w[4], w[5] = rho, rho * vx, rho * vy, bx, by
        w[3] = pr / (GAMMA - 1.0) + 0.5 * rho * (vx * vx + vy * vy) + 0.5 * (bx * bx + by * by)
    else:
        p, rb = (torch.tensor(a, device=dev).expand(shape) for a in configs.hydrostatic(_axes(rp)[0]))
        bz = 0.01 / math.sqrt(configs.MU0)
        cs = torch.sqrt(GAMMA * p / rb)
        w[0] = noise(1e-3) * rb
        for d in range(nd):
            w[1 + d] = (rb + w[0]) * noise(1e-3) * cs
            w[2 + nd + d] = noise(1e-3) * bz
        w[1 + nd] = noise(1e-3) * p / (GAMMA - 1.0)
        w[2 + 2 * nd] = p / (GAMMA - 1.0) + 0.5 * bz * bz
        w[3 + 2 * nd] = rb
        w[4 + 2 * nd] = bz
    return w, pos


def _direction(case, rp, seed, w):
    """Direction of a tangent run: every evolved field and the background,
    each scaled by the field it belongs to."""
    gen = torch.Generator(device=w.device).manual_seed(int(seed) + 7919)
    nd = rp.ndim
    dw = torch.zeros_like(w)
    for f in range(dw.shape[0]):
        g = _smooth(torch.randn(w.shape[1:], generator=gen, device=w.device, dtype=torch.float64))
        dw[f] = g * (w[f] if f >= 2 + 2 * nd else w[f].abs().mean(dim=tuple(range(nd - 1)), keepdim=True))
    return dw


class _View:
    """An evolved field of an engine's device state as an array (no copy); it
    keeps the engine alive."""

    def __init__(self, eng, field):
        self.eng = eng
        self.__cuda_array_interface__ = {"shape": (eng.N,), "typestr": "<f8", "strides": None, "version": 2,
                                         "data": (eng.device_ptr() + 8 * field * eng.N, False)}


def prepare(case, seed):
    rp = _params(case)
    w, pos = _initial(case, rp, seed)
    eng = Engine(rp, w.cpu().numpy(), pos.cpu().numpy())
    s = {"case": case, "rp": rp, "eng": eng, "views": {}}
    if case["kind"] == "tangent":
        k = 2 + 2 * rp.ndim
        dw = _direction(case, rp, seed, w).cpu().numpy().reshape(w.shape[0], -1)
        eng.tl_begin(dw[:k], dbg=dw[k:])
    elif case["restart"]:
        s["w"] = w[: 2 + 2 * rp.ndim].contiguous()
    return s


def run(s):
    case = s["case"]
    eng = s["eng"]
    if case["kind"] == "tangent":
        eng.tl_step(case["steps"])
        w, dw = eng.tl_get()
        return {"w": list(w), "dw": list(dw)}
    if case["restart"]:
        eng.load_pert(s["w"].data_ptr())
        eng.set_clock(0, s["rp"].qt0)
    eng.step(case["steps"])
    ptr = eng.device_ptr()  # the single-stage scheme alternates between two buffers
    if ptr not in s["views"]:
        s["views"][ptr] = [torch.as_tensor(_View(eng, f), device="cuda") for f in range(eng.npert)]
    return s["views"][ptr]


def work(case):
    """Bytes and FP64/FP32 operations of a pass.  Per cell and stage: the wave
    speeds read every field; the update reads every field, the step's base and
    the Runge-Kutta inputs where they are other arrays, and writes the evolved
    fields.  Tangent runs read and write (value, tangent) pairs and bring both
    to the host."""
    nd = case["ndim"]
    cells = case["n0"] * case["n1"] * case["n2"]
    k, nv = 2 + 2 * nd, 4 + 3 * nd
    stages = 4 if case["rk"] else 1
    values = stages * (nv + nv + k) + (3 * k + 2 * k if case["rk"] else 0)  # base of stages 2-4; two inputs of the sum
    flops = stages * (900 if nd == 2 else 2000)
    if case["kind"] == "tangent":
        return {"bytes": cells * 16.0 * (values * case["steps"] + k), "flops": cells * 2.5 * flops * case["steps"]}
    extra = 2 * k if case["restart"] else 0
    return {"bytes": cells * 8.0 * (values * case["steps"] + extra), "flops": float(cells * flops * case["steps"])}


def tolerance(case):
    """Largest differences from exact() seen: 2e-16 on the stratified states,
    8e-16 on the Orszag-Tang flow (whose smooth regions amplify roundoff
    through the ratio max|d3q|/max|dq|), 5e-9 with FP32 stencils over FP64
    states, 1.2e-7 in their tangents; FP64 sums in another order and longer
    runs of other sizes get room for a few times that."""
    if case["mixed"]:
        return {"rel": 5e-7, "max": 1e-4} if case["kind"] == "tangent" else {"rel": 5e-8, "max": 1e-5}
    if case["problem"] == "orszag_tang":
        return {"rel": 1e-12, "max": 1e-10}
    return {"rel": 1e-14, "max": 1e-11}


# --------------------------------------------------------------------------
# the step in float64 torch


class _Exact:
    def __init__(self, case, rp, pos):
        self.rp, self.nd = rp, rp.ndim
        self.case = case
        self.n = rp.n
        self.per = case["problem"] == "orszag_tang"
        self.dev = pos.device
        axes = _axes(rp)
        self.dx = [torch.tensor(np.gradient(axes[d]), device=self.dev).reshape(
            [-1 if self.nd - 1 - q == d else 1 for q in range(self.nd)]) for d in range(self.nd)]
        self.pos = pos
        self.halo = [self._halo_index(d) for d in range(self.nd)]

    def ax(self, d):
        return self.nd - 1 - d

    def cut(self, a, d, lo, hi):
        return a.narrow(self.ax(d), lo, hi - lo)

    # values one step past the grid along d: the cell at 5 below; above, the
    # cell (or zero) whose padded index a linear index shifted by one cell in
    # every direction of the unpadded grid lands on
    def _halo_index(self, d):
        n = list(self.n) + [1] * (3 - self.nd)
        P = [n[0] + 2, n[1] + 2, n[2] + 2]
        idx = np.meshgrid(*[np.arange(n[q]) if q != d else np.array([n[d]]) for q in range(3)], indexing="ij")
        pc = [idx[q] + 1 for q in range(3)]
        z = [np.minimum(pc[q], n[q] - 1) for q in range(3)]
        if self.nd == 3:
            lin = (pc[2] * P[1] + pc[1]) * P[0] + pc[0]
            shift = n[0] * n[1] + n[0] + 1
            tz = (z[2] * n[1] + z[1]) * n[0] + z[0]
        else:
            lin = pc[1] * P[0] + pc[0]
            shift = n[0] + 1
            tz = z[1] * n[0] + z[0]
        h = lin - shift
        ok = (h >= 0) & (h < n[0] * n[1] * n[2]) & (h >= tz)
        h = np.where(ok, h, 0).transpose(2, 1, 0)
        ok = ok.transpose(2, 1, 0)
        if self.nd == 2:
            h, ok = h[0], ok[0]
        return torch.tensor(h, device=self.dev), torch.tensor(ok, device=self.dev)

    def padded(self, q, d):
        h, ok = self.halo[d]
        top = torch.where(ok, q.reshape(-1)[h.reshape(-1)].reshape(h.shape), torch.zeros((), dtype=q.dtype, device=q.device))
        return torch.cat([q.narrow(self.ax(d), 5, 1), q, top], dim=self.ax(d))

    def full(self, a, d):
        """Values of the cells 2..n-3 along d, zeros on the others."""
        shape = list(a.shape)
        shape[self.ax(d)] = 2
        e = torch.zeros(shape, dtype=a.dtype, device=a.device)
        return torch.cat([e, a, e], dim=self.ax(d))

    def nu(self, q, d, scale):
        """nu at i+1/2 and i-1/2 of the cells 2..n-3 along d (zeros elsewhere),
        held constant by derivatives."""
        p = self.padded(q.detach(), d)
        n = self.n[d]
        c = lambda lo, hi: self.cut(p, d, lo, hi)  # noqa: E731
        d1 = (c(1, n + 2) - c(0, n + 1)).abs()  # interfaces 0..n
        d3 = (3.0 * (c(2, n + 1) - c(1, n)) - (c(3, n + 2) - c(0, n - 1))).abs()  # interfaces 1..n-1
        k = n - 3  # interfaces 2..n-2
        m5 = self.cut(d1, d, 0, k)
        for o in range(1, 5):
            m5 = torch.maximum(m5, self.cut(d1, d, o, o + k))
        m3 = self.cut(d3, d, 0, k)
        for o in range(1, 3):
            m3 = torch.maximum(m3, self.cut(d3, d, o, o + k))
        ratio = torch.where(m5 > 0, m3 / torch.where(m5 > 0, m5, torch.ones_like(m5)), torch.zeros_like(m5))
        dxk = self.cut(self.dx[d], d, 2, n - 2) * scale
        return self.full(dxk * self.cut(ratio, d, 1, k), d), self.full(dxk * self.cut(ratio, d, 0, k - 1), d)

    def shift(self, a, d, o):
        """a at i+o (wrapped: only cells 2..n-3 are used)."""
        return torch.roll(a, -o, self.ax(d))

    def layers(self, a, d, count):
        """a with the first and last `count` interior layers along d zeroed
        (not on periodic grids)."""
        if self.per:
            return a
        m = torch.ones(self.n[d], dtype=a.dtype, device=self.dev)
        m[: 2 + count] = 0
        m[self.n[d] - 2 - count:] = 0
        return a * m.reshape(self.dx[d].shape)

    def inner(self, a):
        """a on interior cells, zero on ghosts."""
        m = torch.zeros(a.shape, dtype=a.dtype, device=a.device)
        m[tuple(slice(2, -2) for _ in range(self.nd))] = 1
        return a * m

    def grad4(self, a, d):
        s = lambda o: self.shift(a, d, o)  # noqa: E731
        return self.layers(((8.0 * s(1) - 8.0 * s(-1)) + (s(-2) - s(2))) / (12.0 * self.dx[d]), d, 2)

    def speeds(self, w):
        nd, g = self.nd, GAMMA
        rt = w[0] + w[3 + 2 * nd]
        m, b, bb = w[1: 1 + nd], w[2 + nd: 2 + 2 * nd], w[4 + 2 * nd:]
        mm, b2, bb2, bbb = (m * m).sum(0), (b * b).sum(0), (bb * bb).sum(0), (b * bb).sum(0)
        pk = (g - 1) * (w[1 + nd] - 0.5 * mm / rt - 0.5 * b2 - bbb)
        cs2 = g * (pk + (g - 1) * (w[2 + 2 * nd] - 0.5 * bb2)) / rt
        cf = (b2 + bb2 + 2.0 * bbb) / rt + cs2
        out = []
        for d in range(nd):
            bt = bb[d] + b[d]
            c = torch.sqrt(0.5 * (cf + torch.sqrt(cf * cf - 4.0 * cs2 * bt * bt / rt))) + (m[d] / rt).abs()
            out.append(torch.maximum(c, torch.sqrt(cs2)).max().detach())
        return out

    def dt_of(self, cm):
        rp = self.rp
        if rp.moddton != 1:
            return torch.tensor(rp.dt, dtype=torch.float64, device=self.dev)
        t = rp.courant / torch.clamp(cm[-1] / min(rp.dx), min=1e-12)
        cap = torch.full_like(t, rp.dt)
        return torch.where((t > 1e-12) & (t < cap), t, cap)

    def rhs(self, w, cm):
        nd, g, rp = self.nd, GAMMA, self.rp
        E = 1 + nd
        rho, e, eb, rb = w[0], w[E], w[2 + 2 * nd], w[3 + 2 * nd]
        m = [w[1 + d] for d in range(nd)]
        b = [w[2 + nd + d] for d in range(nd)]
        bb = [w[4 + 2 * nd + d] for d in range(nd)]
        rt = rho + rb
        v = [x / rt for x in m]
        dot = lambda x, y: sum(p * q for p, q in zip(x, y))  # noqa: E731
        mm, b2, bbb, bb2 = dot(m, m), dot(b, b), dot(b, bb), dot(bb, bb)
        pt = (g - 1) * (e - 0.5 * mm / rt) - (g - 2) * (bbb + 0.5 * b2)
        acc = [torch.zeros_like(rho) for _ in range(2 + 2 * nd)]
        for d in range(nd):
            F = [v[d] * rt]
            F[0] = v[d] * rho + rb * v[d]
            for f in range(nd):
                F.append(v[d] * m[f] - (b[f] * bb[d] + bb[f] * b[d]) - b[f] * b[d] + (pt if f == d else 0.0))
            F.append(v[d] * e + v[d] * pt - b[d] * dot(bb, v) - bb[d] * dot(b, v) + v[d] * eb - b[d] * dot(b, v))
            for f in range(nd):
                F.append(None if f == d else v[d] * b[f] - (b[d] + bb[d]) * v[f] + bb[f] * v[d])
            for f, x in enumerate(F):
                if x is not None:
                    acc[f] = acc[f] - self.grad4(x, d)
        ptb = (g - 1) * eb - 0.5 * (g - 2) * bb2
        for f in range(nd):
            gr = [self.grad4(v[f], d) for d in range(nd)]
            acc[E] = acc[E] - ptb * gr[f] + sum(bb[d] * bb[f] * gr[d] for d in range(nd))
        chyp = rp.to_c().chyp
        sides = lambda q, d: (self.layers((self.shift(q, d, 1) - q) / self.dx[d], d, 1),  # noqa: E731
                              self.layers((q - self.shift(q, d, -1)) / self.dx[d], d, 1))
        mid = lambda q, d: self.layers((self.shift(q, d, 1) - self.shift(q, d, -1)) / (2.0 * self.dx[d]), d, 1)  # noqa: E731
        face = lambda q, d, o: 0.5 * (q + self.shift(q, d, o))  # noqa: E731
        qe = e - 0.5 * (b2 + mm / rt)
        for f, q in ((0, rho), (E, qe)):
            for d in range(nd):
                nr, nl = self.nu(q, d, cm[d] * chyp[f])
                gr, gl = sides(q, d)
                acc[f] = acc[f] + (nr * gr - nl * gl) / self.dx[d]
        for f in range(nd):
            for d in range(nd):
                nr, nl = self.nu(v[f], d, cm[d] * chyp[1 + f])
                gr, gl = sides(v[f], d)
                weight = 1.0 if d == f else 0.5
                acc[1 + f] = acc[1 + f] + weight * (face(rt, d, 1) * nr * gr - face(rt, d, -1) * nl * gl) / self.dx[d]
                acc[E] = acc[E] + weight * (face(m[f], d, 1) * nr * gr - face(m[f], d, -1) * nl * gl) / self.dx[d]
                if d != f:
                    t6 = self.inner(mid(v[f], d) * (nr + nl) * 0.25)
                    acc[1 + d] = acc[1 + d] + mid(rt * t6, f)
                    acc[E] = acc[E] + mid(t6 * m[d], f)
        for f in range(nd):
            for d in range(nd):
                if d == f:
                    continue
                q = b[f]
                nr, nl = self.nu(q, d, cm[d] * chyp[2 + nd + f])
                gr, gl = sides(q, d)
                t3 = self.inner(mid(q, d) * (nr + nl) * 0.5)
                acc[2 + nd + d] = acc[2 + nd + d] - mid(t3, f)
                acc[E] = acc[E] - mid(t3 * b[d], f)
                acc[2 + nd + f] = acc[2 + nd + f] + (gr * nr - gl * nl) / self.dx[d]
                acc[E] = acc[E] + (face(q, d, 1) * gr * nr - face(q, d, -1) * gl * nl) / self.dx[d]
        for d in range(nd):
            if rp.g[d] != 0.0:
                acc[1 + d] = acc[1 + d] + rp.g[d] * rho
                acc[E] = acc[E] + rho * rp.g[d] * m[d] / rt
        return acc

    def source(self, out, rb, h, qt):
        rp, nd = self.rp, self.nd
        dv, x = rp.drv, self.pos
        E = 1 + nd
        if self.case["driver"] == "vertical" and not self.per:
            s = torch.exp(-((x[0] - dv[2]) / dv[5]) ** 2)
            for d in range(1, nd):
                s = s * torch.exp(-((x[d] - dv[2 + d]) / dv[6]) ** 2)
            v = dv[0] * s * math.sin(2.0 * math.pi * qt / dv[1])
            rt = out[0] + rb
            out[1] = out[1] + h * v * rt
            out[E] = out[E] + 0.5 * h * v * v * rt
        elif self.case["driver"] == "torsional" and nd == 3:
            z, xp, yp = x[0] - dv[2], x[1] - dv[3], x[2] - dv[4]
            s = torch.exp(-(z / dv[5]) ** 2) * torch.exp(-(xp / dv[6]) ** 2) * torch.exp(-(yp / dv[7]) ** 2) * dv[1]
            vx, vy = dv[0] * yp / dv[9] * s, -dv[0] * xp / dv[8] * s
            rt = out[0] + rb
            out[2] = out[2] + h * vx * rt
            out[3] = out[3] + h * vy * rt
            out[E] = out[E] + 0.5 * h * (vx * vx + vy * vy) * rt
        return out

    def ghosts(self, a):
        """Ghost layers of one field, direction after direction."""
        for d in range(self.nd):
            n, i = self.n[d], torch.arange(self.n[d], device=self.dev)
            if self.per:
                i[:2], i[-2:] = i[:2] + n - 4, i[-2:] - (n - 4)
            else:
                i[0], i[1], i[n - 1], i[n - 2] = 4, 3, n - 5, n - 4
            a = a.index_select(self.ax(d), i)
        return a

    def steps(self, w):
        rp, nd = self.rp, self.nd
        k = 2 + 2 * nd
        cur, bg, qt = [self.ghosts(w[f]) for f in range(k)], w[k:], rp.qt0
        for _ in range(self.case["steps"]):
            qt = qt + rp.dt
            dt = None

            def stage(win, frac):
                nonlocal dt
                full = torch.cat([torch.stack(win), bg])
                cm = self.speeds(full)
                if dt is None:
                    dt = self.dt_of(cm)
                acc = self.rhs(full, cm)
                out = [cur[f] + frac * dt * acc[f] for f in range(k)]
                return self.source(out, bg[1], frac * dt, qt)

            if not self.case["rk"]:
                cur = [self.ghosts(x) for x in stage(cur, 1.0)]
                continue
            w1 = [self.ghosts(x) for x in stage(cur, 0.5)]
            w2 = [self.ghosts(x) for x in stage(w1, 0.5)]
            w3 = [self.ghosts(x) for x in stage(w2, 1.0)]
            o = stage(w3, 1.0 / 6.0)
            cur = [self.ghosts(o[f] + (w1[f] + 2.0 * w2[f] + w3[f] - 4.0 * cur[f]) / 3.0) for f in range(k)]
        return torch.stack(cur)


def exact(case, seed):
    rp = _params(case)
    w, pos = _initial(case, rp, seed)
    x = _Exact(case, rp, pos)
    nd = rp.ndim
    k = 2 + 2 * nd
    with torch.no_grad():
        if case["kind"] == "forward":
            out = x.steps(w)
            return [out[f].reshape(-1) for f in range(k)]
    dw = _direction(case, rp, seed, w)
    val, tan = torch.func.jvp(x.steps, (w,), (dw,))
    return {"w": [a.reshape(-1).cpu().numpy() for a in val], "dw": [a.reshape(-1).cpu().numpy() for a in tan]}
