"""What a user of this library has it do, as cases that can be timed and compared.

A case is a dict of plain values.  Four kinds:

``step``   ``Channel.step(n)``: the main loop between two checks, outputs or
           statistics samples of a run (the driver's default).
``calls``  one time step through the reference's module routines, one call for
           each (the driver with ``fused_step: false``; programs that put work of
           their own between the routines).
``les``    ``Channel.step(n)`` of a coarse run with a learned closure attached.
``train``  Adam steps of the closure's network, one for each of the snapshots.

The velocity and pressure fields come back whole, halo cells included, as views
of the context's device buffers; training returns the parameters.

``exact`` restates each path in 64 bits with plain torch: the staggered
finite-volume tendency, Heun's two stages, the Poisson solve by FFT and Thomas
elimination, the projection, the forcing and the boundary rules.
"""
import math

import numpy as np
import torch

import powerllel_channel_sycl_amd as pll

DEV = "cuda:0"
WAVES = 0.2  # amplitude of each large wave of the initial state, in bulk velocities
PI = math.pi
NIN, NPAD, NH = 10, 16, 64  # the closure's network: 10 (padded to 16) -> 64 -> 64 -> 1


def _grid(name, kind, nx, ny, nz, lx, ly, stretch, re, dt, precision, steps):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, stretch=stretch, re=re,
                dt=dt, precision=precision, steps=steps)


def listed():
    return [
        # the smallest channel that is run in earnest: a set-up check, bound by launches
        _grid("step 24x20x12 fp64", "step", 24, 20, 12, 2 * PI, PI, 1.5, 2800.0, 2e-3, "fp64", 10),
        # the Re_tau~180 minimal channel
        _grid("step 64x64x64 fp64", "step", 64, 64, 64, 2 * PI, PI, 1.5, 2800.0, 2e-3, "fp64", 10),
        # the default grid, one step for each call: a program that looks at every step
        _grid("step1 128x128x128 fp64", "step", 128, 128, 128, 4 * PI, 2 * PI, 1.5, 2800.0, 1e-3,
              "fp64", 1),
        # the Re_tau~180 production grid
        _grid("step 256x192x128 fp64", "step", 256, 192, 128, 4 * PI, 2 * PI, 1.5, 2800.0, 1e-3,
              "fp64", 10),
        # the same grid through the module routines
        _grid("calls 256x192x128 fp64", "calls", 256, 192, 128, 4 * PI, 2 * PI, 1.5, 2800.0, 1e-3,
              "fp64", 1),
        # sizes that are no power of two in any direction (100 = 4*5*5, 90 = 2*3*3*5)
        _grid("step 200x90x176 fp64", "step", 200, 90, 176, 2 * PI, PI, 1.5, 2800.0, 2e-3, "fp64",
              10),
        # the fine run of the closure workflow between two snapshots
        _grid("step 384x256x192 fp32", "step", 384, 256, 192, 2 * PI, PI, 1.5, 6875.0, 4e-3,
              "fp32_mixed", 50),
        # the Re_tau~550 grid in both precisions, at the time step of a statistics run
        _grid("step 768x384x384 fp64", "step", 768, 384, 384, 2 * PI, PI, 1.8, 10000.0, 2e-3,
              "fp64", 10),
        _grid("step 768x384x384 fp32", "step", 768, 384, 384, 2 * PI, PI, 1.8, 10000.0, 2e-3,
              "fp32_mixed", 10),
        # the largest: the Re_tau~1000 grid, 604 million points
        _grid("step 1536x768x512 fp32", "step", 1536, 768, 512, 2 * PI, PI, 2.0, 20000.0, 1e-3,
              "fp32_mixed", 4),
        # the closure workflow's coarse run between two statistics samples
        _grid("les 96x64x64 fp64", "les", 96, 64, 64, 2 * PI, PI, 1.5, 6875.0, 8e-3, "fp64", 25),
        # its training: snapshots of 96 x 64 x 64 samples
        dict(name="train 4x393216", kind="train", samples=96 * 64 * 64, snapshots=4, lr=1e-3),
    ]


def _smooth(lo, hi):
    """Even products of 2, 3 and 5 whose half is one too, lo..hi."""
    out = []
    for n in range(lo + lo % 2, hi + 1, 2):
        m = n // 2
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            out.append(n)
    return out


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: x and y of every length the transforms
    take, z any even number."""
    kind = rng.choice(["step"] * 7 + ["calls", "les", "train"])
    if kind == "train":
        return dict(kind="train", samples=_log_int(rng, 1000, 393216), snapshots=rng.randint(1, 4),
                    lr=1e-3)

    def near(sizes, x):
        return min(sizes, key=lambda n: abs(math.log(n / x)))
    top = dict(step=(768, 384, 512), calls=(512, 384, 256), les=(192, 128, 128))[kind]
    while True:
        scale = math.exp(rng.uniform(math.log(0.05), 0.0))
        nx, ny, nz = (t * min(1.0, scale * math.exp(rng.uniform(-0.7, 0.7))) for t in top)
        nx, ny = near(_smooth(12, top[0]), nx), near(_smooth(10, top[1]), ny)
        nz = max(8, 2 * int(nz / 2))
        if nx * ny * nz <= 40_000_000:
            break
    steps = 1 if kind == "calls" else rng.choice([1, 5, 10, 25])
    while steps > 1 and nx * ny * nz * steps > 300_000_000:
        steps = max(1, steps // 2)
    stretch, re = rng.choice([1.5, 1.8]), rng.choice([2800.0, 6875.0, 10000.0])
    lx, ly = rng.choice([(2 * PI, PI), (4 * PI, 2 * PI)])
    dzmin = min(_dzf(nz, stretch)[1:-1])
    dt = min(0.15 * lx / nx, 0.15 * ly / ny, 0.15 * re * dzmin * dzmin, 8e-3)
    dt = float("%.2g" % dt)
    precision = rng.choice(["fp64", "fp32_mixed"]) if kind == "step" else "fp64"
    c = _grid("", kind, nx, ny, nz, lx, ly, stretch, re, dt, precision, steps)
    del c["name"]
    return c


# ---- inputs -----------------------------------------------------------------------

def _dzf(nz, stretch, lz=2.0):
    """Cell heights 0..nz+1 of the tanh mesh; a ghost cell has its neighbour's."""
    zf = [0.5 * (1.0 + math.tanh((k / nz - 0.5) * stretch) / math.tanh(0.5 * stretch))
          for k in range(1, nz + 1)]
    zf = [0.0] + zf
    dz = [lz * (zf[k] - zf[k - 1]) for k in range(1, nz + 1)]
    return [dz[0]] + dz + [dz[-1]]


def _fill(case, seed, views):
    """A channel profile with unit bulk velocity, a few large waves and 10 %
    noise in u, v and w, written to the interior of the three views (at their
    own precision), some planes at a time to keep the temporaries small."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    dz = torch.tensor(_dzf(nz, case["stretch"]), dtype=torch.float64)[1:-1]
    zc = torch.cumsum(dz, 0) - 0.5 * dz
    prof = 1.5 * (1.0 - (zc - 1.0) ** 2)
    prof = (prof / (prof * dz).sum() * 2.0).to(DEV)
    env = (1.0 - (zc - 1.0) ** 2).to(DEV)
    x = torch.arange(nx, device=DEV, dtype=torch.float64) * (2 * PI / nx)
    y = torch.arange(ny, device=DEV, dtype=torch.float64) * (2 * PI / ny)
    for d, view in enumerate(views):
        ph = torch.rand(6, generator=gen, device=DEV, dtype=torch.float64) * 2 * PI
        wave = sum(torch.cos((m + 1) * y + ph[2 * m])[:, None] *
                   torch.cos((m + 1) * x + ph[2 * m + 1])[None] for m in range(3))
        for k in range(0, nz, 32):
            e = min(nz, k + 32)
            f = 0.2 * (torch.rand((e - k, ny, nx), generator=gen, device=DEV,
                                  dtype=torch.float64) - 0.5)
            f += WAVES * env[k:e, None, None] * wave
            if d == 0:
                f += prof[k:e, None, None]
            view[1 + k:1 + e, 1:-1, 1:-1] = f.to(view.dtype)


class _Buffer:
    """A device buffer of a context as torch sees it; keeps its owner alive."""

    def __init__(self, owner, ptr, shape, elem):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f%d" % elem,
                                             data=(ptr, False), version=2)


def _view(state, field):
    """The current device buffer of a field (a step swaps buffers)."""
    import ctypes
    ch, ptr, elem = state["channel"], state["ptr"], state["elem"]
    rc = state["lib"].pll_field_device_ptr(ch._h, pll.FIELDS[field], ctypes.byref(ptr),
                                           ctypes.byref(elem))
    if rc:
        raise RuntimeError("pll_field_device_ptr failed")
    got = state["views"].get(ptr.value)
    if got is None:
        buf = _Buffer(ch, ptr.value, ch.field_shape, elem.value)
        got = state["views"][ptr.value] = torch.as_tensor(buf, device=DEV)
    return got


def _net_params(seed):
    """W1[16][64] (rows 10..15 zero), b1, W2[64][64], b2, W3[64], b3."""
    r = np.random.default_rng(int(seed))
    w1 = np.zeros((NPAD, NH))
    w1[:NIN] = r.standard_normal((NIN, NH)) * math.sqrt(2.0 / NIN)
    w2 = r.standard_normal((NH, NH)) * math.sqrt(2.0 / NH)
    w3 = r.standard_normal(NH) * math.sqrt(1.0 / NH)
    b = 0.05 * r.standard_normal(2 * NH + 1)
    return np.concatenate([w1.ravel(), b[:NH], w2.ravel(), b[NH:2 * NH], w3, b[2 * NH:]]).astype(
        np.float32)


def _scales(case):
    """Feature and eddy-viscosity scales from the friction velocity of the
    usual correlation Re_tau = 0.09 (2 re)^0.88."""
    re = case["re"]
    utau = 0.09 * (2.0 * re) ** 0.88 / re
    return 1.0 / (re * utau * utau), utau * re / 100.0, 1.0 / re


def _samples(case, seed):
    """Normalised gradients and wall distances with labels that depend on them."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    out = []
    for _ in range(case["snapshots"]):
        x = torch.randn((case["samples"], NIN), generator=gen, device=DEV) * 0.3
        x[:, 9] = torch.rand(case["samples"], generator=gen, device=DEV) * 4.0
        noise = torch.rand(case["samples"], generator=gen, device=DEV)
        y = torch.relu(x[:, 0] * x[:, 4] + x[:, 2].abs() - 0.2 + 0.3 * noise)
        out.append((x.contiguous(), y.contiguous()))
    return out


def _channel(case):
    return pll.Channel(case["nx"], case["ny"], case["nz"], case["lx"], case["ly"], 2.0, case["re"],
                       case["dt"], np.array(_dzf(case["nz"], case["stretch"])),
                       precision=case["precision"])


def prepare(case, seed):
    import ctypes
    if case["kind"] == "train":
        net = pll.Closure(seed=1)
        net.set_params(_net_params(seed))
        data = _samples(case, seed)
        torch.cuda.synchronize()  # the samples are made on torch's stream
        return dict(kind="train", net=net, data=data, n=case["samples"], lr=case["lr"])
    ch = _channel(case)
    state = dict(kind=case["kind"], channel=ch, steps=case["steps"], views={},
                 lib=pll.load_library(), ptr=ctypes.c_void_p(), elem=ctypes.c_int())
    _fill(case, seed, [_view(state, f) for f in "uvw"])
    torch.cuda.synchronize()  # the fields are filled on torch's stream
    ch.updateBoundVel(0)
    ch.updateBoundP()
    if case["kind"] == "les":
        net = pll.Closure(seed=1)
        net.set_params(_net_params(seed))
        net.set_scales(*_scales(case))
        ch.attach_closure(net)
    ch.synchronize()
    return state


def run(state):
    if state["kind"] == "train":
        net, n, lr = state["net"], state["n"], state["lr"]
        for x, y in state["data"]:
            net.train_step(x.data_ptr(), y.data_ptr(), n, lr)
        return net.params()
    ch = state["channel"]
    if state["kind"] == "calls":
        for _ in range(state["steps"]):
            ch.timeIntVelRK1()
            ch.updateBoundVel(1)
            ch.timeIntVelRK2()
            ch.updateBoundVel(0)
            ch.calcRHS()
            ch.execute_poisson_solver()
            ch.updateBoundP()
            ch.correctVel()
            ch.forceVel()
            ch.updateBoundVel(0)
    else:
        ch.step(state["steps"])
    return {f: _view(state, f) for f in ("u", "v", "w", "p")}


def work(case):
    if case["kind"] == "train":
        n = case["samples"] * case["snapshots"]
        # forward and backward products of the network; features and label read once
        return {"bytes": 4.0 * (NIN + 1) * n, "flops": 6.0 * (NIN * NH + NH * NH + NH) * n}
    pts, steps = float(case["nx"]) * case["ny"] * case["nz"], case["steps"]
    e = 8 if case["precision"] == "fp64" else 4
    # a step reads u, v, w and writes u, v, w, p; two stages of about 110
    # operations, two real transforms each way, an elimination and a projection
    fft = 2.0 * 2.5 * (math.log2(case["nx"]) + math.log2(case["ny"]))
    flops = 220.0 + fft + 10.0 + 20.0
    if case["kind"] == "les":
        flops += 2 * 2.0 * (NIN * NH + NH * NH + NH)
    return {"bytes": 7.0 * e * pts * steps, "flops": flops * pts * steps}


# ---- the same in 64 bits ------------------------------------------------------------
# Fields are (nz+2, ny, nx): periodic in x and y, one ghost plane at each wall.

def _e(a):
    return torch.roll(a, -1, -1)


def _w(a):
    return torch.roll(a, 1, -1)


def _n(a):
    return torch.roll(a, -1, -2)


def _s(a):
    return torch.roll(a, 1, -2)


class _Exact:
    def __init__(self, case):
        self.c = case
        nx, ny, nz = self.n = case["nx"], case["ny"], case["nz"]
        self.dx, self.dy = case["lx"] / nx, case["ly"] / ny
        dz = torch.tensor(_dzf(nz, case["stretch"]), dtype=torch.float64, device=DEV)
        col = lambda a: a[:, None, None]  # noqa: E731
        self.dz = dz
        self.dzc = 0.5 * (dz[1:] + dz[:-1])  # face k between cells k and k+1, k = 0..nz
        self.ci, self.fi = col(1.0 / self.dzc), col(1.0 / dz)
        self.lo, self.up = col(dz[:-1]), col(dz[1:])
        self.nu, self.dt = 1.0 / case["re"], case["dt"]

    def walls(self, u, v, w):
        for a in (u, v):
            a[0] = -a[1]
            a[-1] = -a[-2]
        w[0] = 0.0
        w[-2:] = 0.0

    def tendency(self, u, v, w):
        dxi, dyi, nu = 1.0 / self.dx, 1.0 / self.dy, self.nu
        out = []
        ut = (u[:-1] * self.up + u[1:] * self.lo) * self.ci  # twice the face value, k = 0..nz
        vt = (v[:-1] * self.up + v[1:] * self.lo) * self.ci
        fi = self.fi[1:-1]

        def lap(a, az):
            c = a[1:-1]
            return nu * ((_e(c) - 2 * c + _w(c)) * dxi * dxi + (_n(c) - 2 * c + _s(c)) * dyi * dyi + az)

        a = u[1:-1]
        f = (a + _e(a)) ** 2
        conv = (f - _w(f)) * dxi
        f = (a + _n(a)) * (v[1:-1] + _e(v[1:-1]))
        conv += (f - _s(f)) * dyi
        f = ut * (w[:-1] + _e(w[:-1]))
        conv += (f[1:] - f[:-1]) * fi
        g = (u[1:] - u[:-1]) * self.ci
        out.append(lap(u, (g[1:] - g[:-1]) * fi) - 0.25 * conv)

        a = v[1:-1]
        f = (u[1:-1] + _n(u[1:-1])) * (a + _e(a))
        conv = (f - _w(f)) * dxi
        f = (a + _n(a)) ** 2
        conv += (f - _s(f)) * dyi
        f = vt * (w[:-1] + _n(w[:-1]))
        conv += (f[1:] - f[:-1]) * fi
        g = (v[1:] - v[:-1]) * self.ci
        out.append(lap(v, (g[1:] - g[:-1]) * fi) - 0.25 * conv)

        a, ci = w[1:-1], self.ci[1:]
        f = ut[1:] * (a + _e(a))
        conv = (f - _w(f)) * dxi
        f = vt[1:] * (a + _n(a))
        conv += (f - _s(f)) * dyi
        f = (w[:-1] + w[1:]) ** 2
        conv += (f[1:] - f[:-1]) * ci
        g = (w[1:] - w[:-1]) * self.fi[1:]
        out.append(lap(w, (g[1:] - g[:-1]) * ci) - 0.25 * conv)
        return out

    def nut(self, u, v, w, net, scales):
        """The eddy viscosity of every cell with the network's weights rounded
        to bfloat16 (the network's own type) and everything else in 64 bits."""
        dxi, dyi = 1.0 / self.dx, 1.0 / self.dy
        gs, ys, nus = scales
        nx, ny, nz = self.n
        hz = (0.5 / (self.dzc[1:] + self.dzc[:-1]))[:, None, None]
        zc = torch.cumsum(self.dz[1:-1], 0) - 0.5 * self.dz[1:-1]
        sign = torch.where(zc < 1.0, 1.0, -1.0)[:, None, None]
        uc, vc, wc = u + _w(u), v + _s(v), w[1:] + w[:-1]
        wc = wc[:-1]
        um, vm = uc[1:-1], vc[1:-1]
        g = [(u[1:-1] - _w(u[1:-1])) * dxi, (_n(um) - _s(um)) * 0.25 * dyi,
             (uc[2:] - uc[:-2]) * hz * sign, (_e(vm) - _w(vm)) * 0.25 * dxi,
             (v[1:-1] - _s(v[1:-1])) * dyi, (vc[2:] - vc[:-2]) * hz * sign,
             (_e(wc) - _w(wc)) * 0.25 * dxi * sign, (_n(wc) - _s(wc)) * 0.25 * dyi * sign,
             (w[1:-1] - w[:-2]) * self.fi[1:-1]]
        x = [(a * gs).reshape(-1) for a in g]
        yw = torch.minimum(zc, 2.0 - zc) * ys
        x.append(yw[:, None, None].expand(nz, ny, nx).reshape(-1))
        o, _, _, _ = _forward(net, torch.stack(x, 1))
        return nus * torch.nn.functional.softplus(o, threshold=40.0).reshape(nz, ny, nx)

    def stress(self, u, v, w, nu):
        """The divergence of 2 nu S on the faces: normal stresses at the
        centres, shear stresses on the edges, none on a wall's edges."""
        dxi, dyi = 1.0 / self.dx, 1.0 / self.dy
        c = torch.zeros_like(u)
        c[1:-1] = nu
        edge = 0.25 * (nu + _e(nu) + _n(nu) + _e(_n(nu)))
        txy = edge * ((_n(u[1:-1]) - u[1:-1]) * dyi + (_e(v[1:-1]) - v[1:-1]) * dxi)
        cz = 0.25 * (c[1:] + c[:-1])
        cz[0] = 0.0
        cz[-1] = 0.0
        txz = (cz + _e(cz)) * ((u[1:] - u[:-1]) * self.ci + (_e(w[:-1]) - w[:-1]) * dxi)
        tyz = (cz + _n(cz)) * ((v[1:] - v[:-1]) * self.ci + (_n(w[:-1]) - w[:-1]) * dyi)
        txx = 2 * nu * (u[1:-1] - _w(u[1:-1])) * dxi
        tyy = 2 * nu * (v[1:-1] - _s(v[1:-1])) * dyi
        tzz = 2 * c[1:] * (w[1:] - w[:-1]) * self.fi[1:]
        fi, ci = self.fi[1:-1], self.ci[1:]
        return ((_e(txx) - txx) * dxi + (txy - _s(txy)) * dyi + (txz[1:] - txz[:-1]) * fi,
                (txy - _w(txy)) * dxi + (_n(tyy) - tyy) * dyi + (tyz[1:] - tyz[:-1]) * fi,
                (txz[1:] - _w(txz[1:])) * dxi + (tyz[1:] - _s(tyz[1:])) * dyi +
                (tzz[1:] - tzz[:-1]) * ci)

    def poisson(self, rhs):
        nx, ny, nz = self.n
        ex = 2.0 * (torch.cos(2 * PI * torch.arange(nx // 2 + 1, device=DEV, dtype=torch.float64) / nx) - 1)
        ey = 2.0 * (torch.cos(2 * PI * torch.arange(ny, device=DEV, dtype=torch.float64) / ny) - 1)
        lam = ey[:, None] / self.dy ** 2 + ex[None] / self.dx ** 2
        q = torch.fft.rfft2(rhs)
        dz = self.dz.tolist()
        a = [2.0 / (dz[k + 1] * (dz[k] + dz[k + 1])) for k in range(nz)]
        c = [2.0 / (dz[k + 1] * (dz[k + 2] + dz[k + 1])) for k in range(nz)]
        a[0], c[-1] = 0.0, 0.0
        piv = []
        for k in range(nz):
            b = lam - (a[k] + c[k])
            if k:
                m = a[k] / piv[-1]
                b = b - m * c[k - 1]
                q[k] -= m * q[k - 1]
            piv.append(b)
        piv[-1][0, 0] = 1.0
        q[-1] /= piv[-1]
        q[-1, 0, 0] = 0.0  # the constant of the pressure
        for k in range(nz - 2, -1, -1):
            q[k] = (q[k] - c[k] * q[k + 1]) / piv[k]
        return torch.fft.irfft2(q, s=(ny, nx))

    def step(self, u, v, w, net=None, scales=None):
        dt, dxi, dyi = self.dt, 1.0 / self.dx, 1.0 / self.dy

        def rate(a, b, c):
            t = self.tendency(a, b, c)
            if net is not None:
                t = [x + y for x, y in zip(t, self.stress(a, b, c, self.nut(a, b, c, net, scales)))]
            return t
        one = [torch.zeros_like(u) for _ in range(3)]
        for o, f, t in zip(one, (u, v, w), rate(u, v, w)):
            o[1:-1] = f[1:-1] + dt * t
        self.walls(*one)
        for f, o, t in zip((u, v, w), one, rate(*one)):
            f[1:-1] = 0.5 * (f[1:-1] + o[1:-1] + dt * t)
        del one
        self.walls(u, v, w)
        div = (u[1:-1] - _w(u[1:-1])) * dxi + (v[1:-1] - _s(v[1:-1])) * dyi + \
            (w[1:-1] - w[:-2]) * self.fi[1:-1]
        p = torch.zeros_like(u)
        p[1:-1] = self.poisson(div / dt)
        del div
        p[0] = p[1]
        p[-1] = p[-2]
        pi = p[1:-1]
        u[1:-1] -= dt * dxi * (_e(pi) - pi)
        v[1:-1] -= dt * dyi * (_n(pi) - pi)
        w[1:-1] -= dt * (p[2:] - pi) * self.ci[1:]
        nx, ny, _ = self.n
        u[1:-1] += 1.0 - (u[1:-1].sum((1, 2)) * self.dz[1:-1]).sum() / (2.0 * nx * ny)
        self.walls(u, v, w)
        return p


def _forward(p, x):
    """The network on rows x: its output, and what the backward pass needs."""
    bf = lambda a: a.to(torch.bfloat16).to(torch.float64)  # noqa: E731
    w1, o = bf(p[:NPAD * NH]).reshape(NPAD, NH)[:NIN], NPAD * NH
    b1, o = p[o:o + NH], o + NH
    w2, o = bf(p[o:o + NH * NH]).reshape(NH, NH), o + NH * NH
    b2, o = p[o:o + NH], o + NH
    w3, b3 = bf(p[o:o + NH]), p[o + NH]
    x = bf(x.to(torch.float32))
    h1 = torch.relu(x @ w1 + b1)
    h2 = torch.relu(h1 @ w2 + b2)
    return h2 @ w3 + b3, x, h1, h2


def _exact_train(case, seed):
    p = torch.from_numpy(_net_params(seed)).to(DEV).to(torch.float64)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for t, (xs, y) in enumerate(_samples(case, seed), 1):
        o, x, h1, h2 = _forward(p, xs)
        n = x.shape[0]
        d = 2.0 * (torch.nn.functional.softplus(o, threshold=40.0) - y) / n * torch.sigmoid(o)
        at = NPAD * NH + NH
        w2 = p[at:at + NH * NH].to(torch.bfloat16).to(torch.float64).reshape(NH, NH)
        w3 = p[at + NH * NH + NH:at + NH * NH + 2 * NH].to(torch.bfloat16).to(torch.float64)
        d2 = d[:, None] * w3 * (h2 > 0)
        d1 = (d2 @ w2.T) * (h1 > 0)
        g1 = torch.zeros((NPAD, NH), device=DEV, dtype=torch.float64)
        g1[:NIN] = x.T @ d1
        g = torch.cat([g1.reshape(-1), d1.sum(0), (h1.T @ d2).reshape(-1), d2.sum(0), h2.T @ d,
                       d.sum()[None]])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - case["lr"] * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return p


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if nx * ny * nz > 200_000_000:
        return None  # minutes and most of the card's memory in this form
    dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
    fields = []
    views = [torch.zeros((nz + 2, ny + 2, nx + 2), dtype=dtype, device=DEV) for _ in range(3)]
    _fill(case, seed, views)
    while views:
        fields.append(views.pop(0)[:, 1:-1, 1:-1].to(torch.float64).contiguous())
    ex = _Exact(case)
    u, v, w = fields
    ex.walls(u, v, w)
    net = scales = None
    if case["kind"] == "les":
        net = torch.from_numpy(_net_params(seed)).to(DEV).to(torch.float64)
        scales = _scales(case)
    for _ in range(case["steps"]):
        p = ex.step(u, v, w, net, scales)
    return {f: torch.nn.functional.pad(a[None], (1, 1, 1, 1), mode="circular")[0]
            for f, a in (("u", u), ("v", v), ("w", w), ("p", p))}
