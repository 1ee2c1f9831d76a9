"""What a user of the KMM channel solver has it do, as timed cases.

A case is one program at work: a channel (or an ensemble of channels, or the
closure network) set up and held on the GPU, and one pass of it: a number of
time steps and the read-out of the state into the program's own page-locked
buffers (kmm_get_field), or one call of the network's training.  Sizes are
those of the configurations, tests and benchmark of this repository.

  channel   Navier-Stokes (and scalar, immersed rib, tracers, inertial
            particles, constant mass flux, captured graph) time steps
  fenep     the same with FENE-P conformation transport
  closure   the same with the learned polymer-stress closure
  ensemble  independent channels of uneven size advanced together
  train     Adam steps of the closure network on host training pairs
  grad      loss and gradient of the closure network on one batch

FP64 runs return their state as it is (complex128); mixed-precision runs,
whose transforms and products are FP32, keep their snapshots in FP32
(complex64), half the size on disk.
"""
import ctypes
import math

import numpy as np
import torch

from polymer_dns_amd import ic, kmm

XL = 4.0 * math.pi
SIZES = (22, 128, 128, 128, 128, 6)     # layers of the closure network
POLY = ("c11", "c12", "c13", "c22", "c23", "c33")
# the (nx, nz) grids the plane transforms are built for, and the ny
GRIDS = ((32, 32), (64, 32), (64, 64), (96, 96), (128, 64), (128, 128), (192, 192), (256, 128), (256, 256))
NYS = (32, 48, 64, 80, 96, 128, 192)


def _case(kind, nx, ny, nz, precision, steps, **kw):
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, precision=precision, steps=steps, dt=1e-3, re=2800.0, rtau=180.0,
             scalar=False, rib=False, cmf=False, graph=0, tracers=0, inertial=0)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest channel of the tests: four launches a step, latency
        dict(name="channel_32", **_case("channel", 32, 32, 32, "fp64", 50)),
        # the reference's CPU case at constant mass flux, steps replayed as a captured graph
        dict(name="channel_64_graph", **_case("channel", 64, 64, 64, "fp64", 50, cmf=True, graph=10)),
        # the ragged member sizes of the ensembles, alone, with the scalar
        dict(name="channel_96_mixed", **_case("channel", 96, 80, 96, "mixed", 20, scalar=True)),
        # the headline channel: Re_tau 180, scalar, immersed rib
        dict(name="headline_fp64", **_case("channel", 128, 128, 128, "fp64", 20, scalar=True, rib=True)),
        dict(name="headline_mixed", **_case("channel", 128, 128, 128, "mixed", 20, scalar=True, rib=True)),
        # inertial particles (Maxey-Riley) in a channel
        dict(name="inertial_64", **_case("channel", 64, 64, 64, "fp64", 20, tracers=10000, inertial=1)),
        # the viscoelastic channel, 100 000 tracers
        dict(name="fenep_192_fp64", **_case("fenep", 192, 128, 192, "fp64", 10, dt=1e-4, tracers=100000)),
        dict(name="fenep_192_mixed", **_case("fenep", 192, 128, 192, "mixed", 10, dt=1e-4, tracers=100000)),
        # the Re_tau 395 viscoelastic channel, the largest work
        dict(name="fenep_256_fp64", **_case("fenep", 256, 192, 256, "fp64", 6, dt=1e-4, re=6875.0, rtau=395.0)),
        # the learned closure in the place of the conformation transport
        dict(name="closure_192", **_case("closure", 192, 128, 192, "mixed", 9, dt=1e-4)),
        # sixteen uneven channels (64 x 49 x 64 to 128 x 97 x 128) together
        dict(name="ensemble_16", **_case("ensemble", 128, 96, 128, "mixed", 10, dt=2e-3, members=16, sizes=20261206)),
        # the closure's training: mini-batches of 1024 from 20 000 pairs
        dict(name="train_1024", **_case("train", 0, 0, 0, "mixed", 20, batch=1024, pairs=20000)),
    ]


def _points(c):
    return c["nx"] * (c["ny"] + 1) * c["nz"]


def draw(rng):
    kind = rng.choice(("channel", "channel", "channel", "fenep", "fenep", "closure", "ensemble", "train", "grad"))
    prec = rng.choice(("fp64", "mixed"))
    if kind == "train":
        n = int(2.0 ** rng.uniform(6.0, 12.0))
        return _case(kind, 0, 0, 0, "mixed", rng.randint(2, 30), batch=n, pairs=n * rng.randint(1, 8) + rng.randint(0, 99))
    if kind == "grad":
        return _case(kind, 0, 0, 0, rng.choice(("fp64", "mixed")), 1, batch=int(2.0 ** rng.uniform(5.0, 14.0)), pairs=0)
    if kind == "ensemble":
        return _case(kind, 128, 96, 128, prec, rng.randint(2, 10), dt=rng.uniform(5e-4, 2e-3), members=rng.randint(2, 16),
                     sizes=rng.randint(1, 9999))
    nx, nz = rng.choice(GRIDS if kind == "channel" else GRIDS[:-1])
    ny = rng.choice(NYS if kind == "channel" else NYS[:-1])
    steps = max(1, min(60, int(4e7 / (nx * nz * (ny + 1)) * rng.uniform(0.5, 1.0))))
    if kind != "channel":
        return _case(kind, nx, ny, nz, "mixed" if kind == "closure" else prec, min(steps, 9), dt=rng.uniform(5e-5, 1e-4),
                     tracers=rng.choice((0, 0, 5003, 100000)) if kind == "fenep" else 0)
    part = rng.choice((0, 0, 0, 1001, 30000))
    small = nx * nz <= 128 * 128
    return _case(kind, nx, ny, nz, prec, steps, dt=rng.uniform(2e-4, 8e-4), scalar=rng.random() < 0.5, rib=rng.random() < 0.3,
                 cmf=rng.random() < 0.3, graph=rng.choice((0, 0, 2, 5)), tracers=part,
                 inertial=int(part > 0 and small and rng.random() < 0.5))


# ------------------------------------------------------------------ inputs --
def _embed(a, nx, nz):
    """Modes of a 32 x 32 field in the layout of an nx x nz one."""
    b = np.zeros((nx // 2, nz, a.shape[2]), dtype=np.complex128)
    b[:15, :16] = a[:15, :16]
    b[:15, nz - 15:] = a[:15, 17:]
    return b


def _flow(c, seed, rtau=None):
    """Laminar profile plus a seeded solenoidal perturbation of its lowest modes (5 % of the centre line)."""
    s = ic.seeded_state(32, 32, 32, XL, _zl(c), c["re"], rtau or c["rtau"], seed, amp=0.05, kmax=8)
    st = {}
    for k in ("v", "omy"):
        a = np.zeros((16, 32, c["ny"] + 1), dtype=np.complex128)
        a[:, :, :33] = s[k][:, :, :c["ny"] + 1]
        st[k] = _embed(a, c["nx"], c["nz"])
    st["u0"] = ic.laminar_u0(c["ny"], c["re"], rtau or c["rtau"])[0]
    st["w0"] = np.zeros(c["ny"] + 1)
    if c["scalar"]:
        r = np.random.default_rng(seed)
        sc = np.zeros((16, 32, c["ny"] + 1), dtype=np.complex128)
        sc[1:6, 1:6, :6] = 0.05 * (r.standard_normal((5, 5, 6)) + 1j * r.standard_normal((5, 5, 6)))
        sc[0, 0, 0] = 0.5
        st["scalar"] = _embed(sc, c["nx"], c["nz"])
    return st


def _zl(c):
    return XL / 3.0


def _rib(c):
    """One spanwise rib on the y = +1 wall, 0.1 high and 0.2 long."""
    from polymer_dns_amd.restart import rib_geometry
    y = np.cos(np.arange(c["ny"] + 1) * math.pi / c["ny"])
    mx = 3 * c["nx"] // 2
    return rib_geometry(c["nx"], c["ny"], c["nz"], y_cells=int(np.sum(y >= 0.9)), x_center=int(round(0.4 * mx)),
                        x_width=max(1, int(round(0.2 / (XL / mx)))))


def _channel(c, seed, rtau=None):
    poly = c["kind"] in ("fenep", "closure")
    rt = rtau or c["rtau"]
    kw = dict(xl=XL, zl=_zl(c), re=c["re"], dt=c["dt"], r_tau=rt, precision=int(c["precision"] == "mixed"))
    if c["scalar"]:
        kw.update(scalar=1, diff=0.71, scl_flag=6, deltaT=1.0)
    if c["rib"]:
        kw.update(gain=20.0, ugain=100.0)
    if c["cmf"]:
        kw.update(cmf=1)
    if c["tracers"]:
        kw.update(ap=1e-3)
    if c["inertial"]:
        kw.update(particle_flag=1, ratio=2.0, c_mu=1.0, cd_switch=0, gravity=0.0)
    tpoly = 50.0 * c["re"] / rt ** 2              # Wi_tau 50
    if poly:
        kw.update(polymer=1, zlmax=30.0, tpoly=tpoly, diffpoly=0.5, qbeta=0.9, ipeter=1, itarget=0, crstrt=1, src_start=0)
    ch = kmm.Channel(kmm.make_config(c["nx"], c["ny"], c["nz"], **kw))
    if c["rib"]:
        ch.set_geometry(_rib(c))
    st = _flow(c, seed, rt)
    for k, v in st.items():
        ch.put(k, v)
    if poly:
        mean = ic.shear_equilibrium(st["u0"], tpoly, 30.0, ipeter=1)
        for k, v in ic.conformation_state(32, c["ny"], 32, seed + 1, amp=1e-3, mean=mean).items():
            ch.put(k, _embed(v, c["nx"], c["nz"]))
    if c["tracers"]:
        r = np.random.default_rng(seed + 2)
        n = c["tracers"]
        ch.set_particles(r.uniform(0, XL, n), r.uniform(-0.95, 0.95, n), r.uniform(0, _zl(c), n))
    ch.startup()
    if c["graph"]:
        ch.set_graph(c["graph"])
    return ch


def _buffers(c, ch):
    """Page-locked read-out buffers of the fields a snapshot holds."""
    names = ["v", "omy"] + (["scalar"] if c["scalar"] else []) + (list(POLY) if c["kind"] == "fenep" else [])
    shape = (ch.nxh, ch.nz, ch.nyp)
    out = {k: torch.empty(shape, dtype=torch.complex128, pin_memory=True) for k in names}
    if c["precision"] == "mixed":
        out = {k: (b, torch.empty(shape, dtype=torch.complex64)) for k, b in out.items()}
    return out


def _pairs(n, seed):
    """Normalised training pairs: 22 features of scale 1 and a smooth 6-component target of them."""
    r = np.random.default_rng(seed)
    X = r.standard_normal((n, 22)).astype(np.float32)
    A = r.standard_normal((22, 6)) / 5.0
    return X, (np.tanh(X @ A) + 0.1 * r.standard_normal((n, 6))).astype(np.float32)


def _net(seed, sd_y=1.0, X=None):
    net = kmm.Mlp(seed=seed)
    net.set_activation("gelu_poly")
    mu, sd = (X.mean(0), X.std(0) + 1e-12) if X is not None else (np.zeros(22), np.ones(22))
    net.set_norm(mu, sd, np.zeros(6), np.full(6, sd_y))
    return net


def prepare(case, seed):
    c = case
    if c["kind"] in ("train", "grad"):
        n = c["pairs"] if c["kind"] == "train" else c["batch"]
        X, T = _pairs(n, seed)
        return dict(case=c, net=_net(seed), X=X, T=T, seed=seed)
    if c["kind"] == "ensemble":
        chans = []
        for m, (nx, ny, nz, rt, s) in enumerate(ic.ensemble_members(c["sizes"], n=c["members"])):
            chans.append(_channel(dict(c, nx=nx, ny=ny, nz=nz), s % 100000 + seed, rt))
        return dict(case=c, chans=chans, bufs=[_buffers(c, ch) for ch in chans])
    ch = _channel(c, seed)
    s = dict(case=c, ch=ch, bufs=_buffers(c, ch))
    if c["kind"] == "closure":
        # a stress history from FENE-P steps, then the network (random weights, a correction
        # small enough for the closed loop to stay near linear extrapolation) takes over
        ch.set_poly_capture(True)
        ch.step(3)
        X, _ = ch.poly_samples(5000, seed=seed)
        s["net"] = _net(seed, 1e-9, X)
        ch.set_closure(s["net"])
        ch.step(3)
    return s


def _read(ch, bufs):
    out = {}
    for k, b in bufs.items():
        host = b[0] if isinstance(b, tuple) else b
        p = ctypes.cast(host.data_ptr(), ctypes.POINTER(ctypes.c_double))
        rc = ch.lib.kmm_get_field(ch.h, kmm.FIELD_ID[k], p)
        if rc:
            raise RuntimeError("kmm_get_field: %d" % rc)
        out[k] = b[1].copy_(host) if isinstance(b, tuple) else host
    return out


def run(state):
    c = state["case"]
    if c["kind"] == "train":
        losses = state["net"].train(state["X"], state["T"], steps=c["steps"], batch=c["batch"], lr=1e-3, seed=state["seed"])
        return {"losses": losses, "params": state["net"].params()}
    if c["kind"] == "grad":
        loss, g = state["net"].grad(state["X"], state["T"], mode=int(c["precision"] == "mixed"))
        return {"loss": np.float32(loss), "grad": g}
    if c["kind"] == "ensemble":
        kmm.ensemble_step(state["chans"], c["steps"])
        return [_read(ch, b) for ch, b in zip(state["chans"], state["bufs"])]
    ch = state["ch"]
    ch.step(c["steps"])
    out = _read(ch, state["bufs"])
    if c["precision"] == "fp64":
        out.update(u0=ch.get("u0"), w0=ch.get("w0"))
    if c["tracers"]:
        t = np.float64 if c["precision"] == "fp64" else np.float32
        out.update({k: v.astype(t, copy=False) for k, v in ch.particles().items() if k != "swirl"})
    return out


# -------------------------------------------------------------------- work --
def _step_work(nx, ny, nz, scalar, kind, mixed):
    """Bytes and operations of a step: the state read and written once, and every field that crosses between
    the wall-normal (whole pencils) and the plane (whole x-z planes) transforms written and read once."""
    G = nx * (ny + 1) * nz
    t = 4 if mixed else 8
    nin, nout = (9, 4) if scalar else (6, 3)
    b = (12 if scalar else 8) * 8.0 + 2 * (nin + nout) * t
    fin, fout, cheb = nin, nout, nin + nout
    if kind == "fenep":
        b += 6 * 6 * 8.0 + 2 * (12 + 3 + 12) * t   # C, c_nm1, str_nm1 in and out; C, dC/dy, Du; c_n, str_n
        fin, fout, cheb = nin + 24, nout + 12, cheb + 15 + 12
    net = 0.0
    if kind == "closure":
        b += 2 * 6 * t + 2 * 6 * 4 * 2.25 * 1.5    # six stresses back; the history on the 3/2 grid in and out
        fin, fout, cheb = nin + 2, nout + 6, cheb + 6
        net = 105472.0 * 2.25 * G
    P, mx, mz = nx // 2 * nz, 1.5 * nx, 1.5 * nz
    fft = lambda n: 5.0 * n * math.log2(n)
    f = (fin + fout) * (ny + 1) * (nx // 2 * fft(mz) + mz * fft(mx) / 2.0)
    f += cheb * P * fft(2 * ny) / 2.0
    f += (4 + (1 if scalar else 0) + (6 if kind == "fenep" else 0)) * P * ny * 30.0 + 2.25 * G * (100 if kind == "fenep" else 30)
    return b * G, f + net


def work(case):
    c = case
    if c["kind"] in ("train", "grad"):
        macs = sum(a * b for a, b in zip(SIZES, SIZES[1:]))
        n, par = c["batch"], 4.0 * (macs + sum(SIZES[1:]))
        k = c["steps"]
        return {"bytes": k * (n * 28 * 4.0 + (6 if c["kind"] == "train" else 2) * par), "flops": k * 6.0 * macs * n}
    mixed = c["precision"] == "mixed"
    if c["kind"] == "ensemble":
        sizes = [m[:3] for m in ic.ensemble_members(c["sizes"], n=c["members"])]
    else:
        sizes = [(c["nx"], c["ny"], c["nz"])]
    by = fl = 0.0
    for nx, ny, nz in sizes:
        b, f = _step_work(nx, ny, nz, c["scalar"], c["kind"], mixed)
        nread = 2 + c["scalar"] + 6 * (c["kind"] == "fenep")
        by += c["steps"] * (b + c["tracers"] * 6 * 8.0 * 2) + nread * 8.0 * nx * (ny + 1) * nz
        fl += c["steps"] * f
    return {"bytes": by, "flops": fl}


# ------------------------------------------------- 64-bit values, plain torch/numpy --
def exact(case, seed):
    c = case
    if c["kind"] == "grad":
        return _exact_grad(c, seed)
    if c["kind"] == "channel" and _points(c) <= 96 * 81 * 96 and not (c["rib"] or c["tracers"]) and c["steps"] <= 60:
        return _ExactChannel(c).run(_flow(c, seed))
    return None


def _exact_grad(c, seed):
    """Loss and gradient by torch autograd in 64 bits, weights and layer inputs rounded to bfloat16 in mode 1
    (the rounding passes the gradient through, as the training does)."""
    X, T = _pairs(c["batch"], seed)
    net = _net(seed)
    Ws, bs = net.unpack()
    net.close()
    bf = (lambda t: t + (t.detach().to(torch.float32).to(torch.bfloat16).double() - t.detach())) if c["precision"] == "mixed" \
        else (lambda t: t)
    Ws = [torch.tensor(w, dtype=torch.float64, requires_grad=True) for w in Ws]
    bs = [torch.tensor(b, dtype=torch.float64, requires_grad=True) for b in bs]
    a = torch.tensor(X, dtype=torch.float64)
    for l, (w, b) in enumerate(zip(Ws, bs)):
        a = bf(a) @ bf(w).T + b
        if l < 4:
            t = torch.clamp(0.5 + a / 5.28, 0.0, 1.0)
            a = a * (t ** 3 * (t * (6.0 * t - 15.0) + 10.0))
    loss = ((a - torch.tensor(T, dtype=torch.float64)) ** 2).sum(1).mean()
    loss.backward()
    g = torch.cat([torch.cat([w.grad.reshape(-1), b.grad]) for w, b in zip(Ws, bs)])
    return {"loss": np.float64(loss.item()), "grad": g.numpy()}


class _ExactChannel:
    """The channel step (Navier-Stokes and scalar) in numpy, 64 bits, with dense matrices in y: the integrated
    Chebyshev tau equations (-D - wn R) u = R f, rows 0 and 1 holding the two boundary conditions."""

    def __init__(self, c):
        self.c = c
        nx, ny, nz = c["nx"], c["ny"], c["nz"]
        self.nxh, self.N, self.nz, self.mx, self.mz = nx // 2, ny + 1, nz, 3 * nx // 2, 3 * nz // 2
        N = self.N
        n = np.arange(N, dtype=np.float64)
        self.kx = (np.arange(nx // 2) * 2.0 * math.pi / XL)[:, None, None]
        kz = np.arange(nz, dtype=np.float64)
        kz[nz // 2:] -= nz
        self.kz = (kz * 2.0 * math.pi / _zl(c))[None, :, None]
        self.k2 = self.kx ** 2 + self.kz ** 2
        R = np.zeros((N, N))
        for j in range(2, N):
            R[j, j - 2] = -(2.0 if j == 2 else 1.0) / (4.0 * j * (j - 1))
            if j <= ny - 2:
                R[j, j] = 1.0 / (2.0 * (j * j - 1))
            if j + 2 <= ny - 2:
                R[j, j + 2] = -1.0 / (4.0 * j * (j + 1))
        self.R, self.sg, self.n2 = R, (-1.0) ** n, n * n
        D = np.zeros((N, N))
        for j in range(N):
            D[j, j + 1::2] = 2.0 * n[j + 1::2]
        D[0] *= 0.5
        self.D = D
        self.c0 = c["re"] / (c["dt"] * 0.5)
        dirichlet = (np.ones(N), self.sg)
        self.H, Hb = self._operator(self.c0, dirichlet)
        self.Pn, _ = self._operator(0.0, dirichlet)
        if c["scalar"]:
            self.S, _ = self._operator(self.c0 * 0.71, (self.n2, -self.sg * self.n2))
        self.G = [self._ap(self.Pn, Hb[:, :, :, b].astype(np.complex128)) for b in (0, 1)]
        jj = np.minimum(np.arange(nz), nz - np.arange(nz))
        self.smooth = (np.exp(-3.0 * (jj / (nz // 2)) ** 10)[:, None] * np.exp(-3.0 * (n / ny) ** 10)[None, :])[None]
        self.dpdx = -(c["rtau"] / c["re"]) ** 2

    def _operator(self, g, rows):
        """(f -> u) and (boundary data -> u) for every pencil; pencils of equal k2 share theirs."""
        wn, back = np.unique(np.round(self.k2[:, :, 0], 12), return_inverse=True)
        M = -np.eye(self.N)[None] - (wn + g)[:, None, None] * self.R[None]
        M[:, 0], M[:, 1] = rows
        if g == 0.0:
            M[0] = np.eye(self.N)
        rhs = np.concatenate([self.R, np.eye(self.N)[:, :2]], axis=1)
        X = np.linalg.solve(M, np.broadcast_to(rhs, (len(wn),) + rhs.shape))[back.reshape(self.k2.shape[:2])]
        return X[..., :self.N], X[..., self.N:]

    @staticmethod
    def _ap(K, f):
        r = np.matmul(K, np.stack([f.real, f.imag], -1))
        return r[..., 0] + 1j * r[..., 1]

    def _d(self, f):
        return f @ self.D.T

    def _dct(self, a):
        return np.fft.fft(np.concatenate([a, a[..., -2:0:-1]], -1), axis=-1)[..., :self.N]

    def _phys(self, a):
        f = a * 0.5
        f[..., 0] *= 2.0
        f[..., -1] *= 2.0
        f = self._dct(f)
        pad = np.zeros((self.mx // 2 + 1, self.mz, self.N), dtype=np.complex128)
        h = self.nz // 2
        pad[:self.nxh, :h] = f[:, :h]
        pad[:self.nxh, self.mz - h:] = f[:, h:]
        return np.fft.irfft(np.fft.ifft(pad, axis=1) * self.mz, n=self.mx, axis=0) * self.mx

    def _spec(self, p):
        f = np.fft.fft(np.fft.rfft(p, axis=0)[:self.nxh], axis=1) / (self.mx * self.mz)
        h = self.nz // 2
        f = self._dct(np.concatenate([f[:, :h], f[:, self.mz - h:]], 1)) / (self.N - 1)
        f[..., 0] *= 0.5
        f[..., -1] *= 0.5
        return self._sym(f)

    def _sym(self, a):
        j = np.arange(1, self.nz // 2)
        a[0, 0] = a[0, 0].real
        a[0, j] = 0.5 * (a[0, j] + np.conj(a[0, self.nz - j]))
        a[0, self.nz - j] = np.conj(a[0, j])
        a[:, self.nz // 2] = 0.0
        return a

    def _terms(self, smooth):
        s, kx, kz = self.s, self.kx, self.kz
        w2 = self.k2.copy()
        w2[0, 0] = 1.0
        dv = self._d(s["v"])
        u = (1j * kx * dv - 1j * kz * s["omy"]) / w2
        w = (1j * kz * dv + 1j * kx * s["omy"]) / w2
        u[0, 0], w[0, 0] = s["u0"], s["w0"]
        ox, oz = self._d(w) - 1j * kz * s["v"], 1j * kx * s["v"] - self._d(u)
        U, V, W, A, B, C = (self._phys(self._sym(a.copy())) for a in (u, s["v"], w, ox, s["omy"], oz))
        h1, h2, h3 = (self._spec(a) for a in (V * C - W * B - self.dpdx, W * A - U * C, U * B - V * A))
        if "scalar" in s:
            q = s["scalar"]
            sn = -(U * self._phys(1j * kx * q) + V * self._phys(self._d(q)) + W * self._phys(1j * kz * q)) + 1.0
            s["sn"] = self._spec(sn) * (self.smooth if smooth else 1.0)
        if smooth:
            h1, h2, h3 = (a * self.smooth for a in (h1, h2, h3))
        s["h1"], s["h3"] = h1[0, 0].real.copy(), h3[0, 0].real.copy()
        s["fn"] = self._sym(-self.k2 * h2 - self._d(1j * (kz * h3 + kx * h1)))
        s["gn"] = self._sym(1j * (kz * h1 - kx * h3))

    def _rhs(self, q, n, m, var=1.0):
        return -self.c0 * var * q - self.c["re"] * var * (3.0 * n - m) + self.k2 * q - self._d(self._d(q))

    def _mean(self, q, n, m):
        f = -self.c0 * q - self.c["re"] * (3.0 * n - m) - self._d(self._d(q))
        return self.H[0, 0] @ f

    def run(self, st):
        s = self.s = {k: np.array(v) for k, v in st.items()}
        for k in ("v", "omy", "scalar"):
            if k in s:
                self._sym(s[k])
        s["v"][0, 0] = s["omy"][0, 0] = 0.0
        n = np.arange(0, self.N, 2)
        bulk = lambda a: float((a[::2] / (1.0 - n * n.astype(np.float64))).sum())
        target = bulk(s["u0"])
        self._terms(False)
        old = {k: s[k].copy() for k in ("fn", "gn", "h1", "h3", "sn") if k in s}
        for _ in range(self.c["steps"]):
            new = {k: s[k].copy() for k in old}
            if "sn" in s:
                s["scalar"] = self._ap(self.S, self._rhs(s["scalar"], s["sn"], old["sn"], 0.71))
            phi = self._d(self._d(s["v"])) - self.k2 * s["v"]
            v = self._ap(self.Pn, self._ap(self.H, self._rhs(phi, s["fn"], old["fn"])))
            g1, g2 = self.G
            t, b = self.n2, -self.sg * self.n2
            a11, a12, a21, a22 = g1 @ t, g2 @ t, g1 @ b, g2 @ b
            det = a11 * a22 - a12 * a21
            det[0, 0] = 1.0
            c1 = -((v @ t) * a22 - (v @ b) * a12) / det
            c2 = -((v @ b) * a11 - (v @ t) * a21) / det
            omy = self._ap(self.H, self._rhs(s["omy"], s["gn"], old["gn"]))
            s["v"] = self._sym(v + c1[..., None] * g1 + c2[..., None] * g2)
            s["omy"] = self._sym(omy)
            s["v"][0, 0] = s["omy"][0, 0] = 0.0
            s["u0"], s["w0"] = self._mean(s["u0"], s["h1"], old["h1"]), self._mean(s["w0"], s["h3"], old["h3"])
            if self.c["cmf"]:
                unit = np.zeros(self.N)
                unit[0] = -2.0 * self.c["re"]
                r = self.H[0, 0] @ unit
                f = (target - bulk(s["u0"])) / bulk(r)
                s["u0"] = s["u0"] + f * r
                self.dpdx -= f
            old = new
            self._terms(True)
        out = {k: s[k] for k in ("v", "omy", "scalar") if k in s}
        if self.c["precision"] == "fp64":
            out.update(u0=s["u0"], w0=s["w0"])
        return {k: torch.from_numpy(np.ascontiguousarray(a)) for k, a in out.items()}
