"""Workloads of the framework through its public entry points (``mwf_amd``).

What a user of Model Waleffe Flow on the GPU has it do:

``run``        a simulation: ``vel_TS`` in blocks of steps, the energy after each
               block (the reference's log line every i_save_rate2 = 50 steps), the
               state at the end (its state file).  From the 64^2-mode parity model
               to the 2048^2-mode M6 box, square and elongated, FP64 and mixed.
``monitor``    one pass of the reference's io_write2files: steps, then energy,
               spectra, velocity profile, turbulence samples, turbulent fraction.
``ensemble``   many members stepped together with tracking on the device, their
               energies and states at the end.
``field``      the nonlinear term of a state and its physical field (host arrays).
``transform``  the transform module on host arrays, both directions.

``tuned`` models are created with ``autotune(1)``, as the Fortran driver and the
benchmark create theirs; the others with the library's default.  Outputs of the
mixed form, whose transforms are FP32, are handed on in single precision.

A model continues from pass to pass, as a simulation does.
"""
import math

import numpy as np
import torch

import mwf_amd as mw

PI = math.pi
BETA = PI / 2
DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64, C128 = torch.float64, torch.complex128


# ----------------------------------------------------------------- the cases

def _run(name, k0, mm, nn, every, blocks, mixed=False, tuned=True, re=200.0, dt=0.02, per=PI / 4, deg=0.0,
         rms=0.3, k0ic=8.0):
    c = dict(kind="run", k0=k0, mm=mm, nn=nn, every=every, blocks=blocks, mixed=mixed, tuned=tuned, re=re, dt=dt,
             per=per, deg=deg, rms=rms, k0ic=k0ic)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the 64^2-mode parity model as a small interactive run: launches and latency
        _run("m4_64", 4, 32, 32, 50, 2, tuned=False, rms=0.1, k0ic=4.0),
        # one medium model by itself
        _run("m6_256", 6, 128, 128, 50, 2),
        # a box made long in x (doubleX/quadX), tilted, mixed form, library defaults
        _run("m4_1024x128_tilted_mixed", 4, 512, 64, 50, 2, mixed=True, tuned=False, deg=24.0),
        # the headline box: 1024^2 modes on a 1536^2 grid
        _run("m4_1024", 4, 512, 512, 50, 4, re=180.0),
        _run("m4_1024_mixed", 4, 512, 512, 50, 4, mixed=True, re=180.0),
        # the largest box: M6, 2048^2 modes on a 3072^2 grid
        _run("m6_2048", 6, 1024, 1024, 25, 2, re=250.0, dt=0.01),
        _run("m6_2048_mixed", 6, 1024, 1024, 25, 2, mixed=True, re=250.0, dt=0.01),
        # the reference's per-save output of a running model, library defaults
        dict(name="monitor_m4_512", kind="monitor", k0=4, mm=256, nn=256, steps=50, tuned=False, re=200.0, dt=0.02,
             per=PI / 4, deg=0.0, rms=0.3, k0ic=8.0, stride=12),
        # lifetime statistics: 256 members of 128^2 modes, Re spread over the transition
        dict(name="ensemble_256_m4_128", kind="ensemble", k0="4", modes="128", members=256, steps=100, every=50,
             mixed=False, tuned=True, re=185.0, spread=35.0, dt=0.02, per=PI / 4, rms=0.25, k0ic=8.0, turb=True),
        # an uneven parameter sweep, M4 and M6 members of 64^2 to 512^2 modes, mixed form
        dict(name="ensemble_48_uneven_mixed", kind="ensemble", k0="4,4,4,6", modes="64,128,256,512", members=48,
             steps=50, every=50, mixed=True, tuned=True, re=225.0, spread=75.0, dt=0.01, per=0.8 * PI,
             rms=0.2, k0ic=8.0, turb=False),
        # field output and the nonlinear term of a stored state
        dict(name="field_m6_512x256", kind="field", k0=6, mm=256, nn=128, mixed=False, tuned=False, re=200.0, dt=0.02,
             per=PI / 4, deg=0.0, rms=0.3, k0ic=8.0),
        # the transform module on the host's arrays
        dict(name="transform_m4_256", kind="transform", k0=4, mm=128, nn=128, mixed=False, tuned=False, re=200.0,
             dt=0.02, per=PI / 4, deg=0.0, rms=0.3, k0ic=8.0),
    ]


def draw(rng):
    kind = rng.choice(["run"] * 5 + ["monitor", "ensemble", "ensemble", "field", "transform"])
    k0 = rng.choice([4, 4, 6])
    mixed = rng.random() < 0.4
    tuned = rng.random() < 0.6
    re = round(rng.uniform(150.0, 300.0), 2)
    dt = rng.choice([0.01, 0.02])
    per = round(PI / 4 * rng.uniform(0.9, 1.3), 4)
    rms = round(rng.uniform(0.05, 0.35), 3)
    deg = rng.choice([0.0, round(rng.uniform(-45.0, 45.0), 1)])

    def size(total):  # powers of two in [16, 1024], their product at most 2^total, up to 1:16
        while True:
            a, b = rng.randint(4, 10), rng.randint(4, 10)
            if a + b <= total and abs(a - b) <= 4:
                return 1 << a, 1 << b

    if kind == "run":
        mm, nn = size(18)
        every = rng.randint(10, 60)
        blocks = rng.randint(1, 3)
        return _run(None, k0, mm, nn, every, blocks, mixed=mixed, tuned=tuned, re=re, dt=dt, per=per, deg=deg, rms=rms,
                    k0ic=rng.choice([4.0, 8.0]))
    if kind == "monitor":
        mm, nn = size(16)
        return dict(kind=kind, k0=k0, mm=mm, nn=nn, steps=rng.randint(20, 60), tuned=tuned, re=re, dt=dt, per=per,
                    deg=deg, rms=rms, k0ic=8.0, stride=rng.choice([4, 6, 8, 12]))
    if kind == "ensemble":
        members = rng.randint(3, 64)
        modes = ",".join(str(x) for x in sorted(rng.sample([32, 64, 128, 256], rng.randint(1, 3))))
        return dict(kind=kind, k0=rng.choice(["4", "6", "4,4,4,6"]), modes=modes, members=members,
                    steps=rng.randint(20, 60), every=rng.randint(5, 20), mixed=mixed, tuned=tuned, re=re, spread=40.0,
                    dt=dt, per=per, rms=rms, k0ic=8.0, turb=not mixed and rng.random() < 0.5)
    mm, nn = size(15)
    return dict(kind=kind, k0=k0, mm=mm, nn=nn, mixed=mixed, tuned=tuned, re=re, dt=dt, per=per, deg=deg, rms=rms,
                k0ic=8.0)


# ------------------------------------------------------------ models, inputs

def _params(c, k0=None, mm=None, nn=None, re=None):
    mm, nn = mm or c["mm"], nn or c["nn"]
    return mw.make_params(k0 or c["k0"], mm, nn, mm * c["per"], nn * c["per"], re or c["re"], c["dt"],
                          thdeg=c.get("deg", 0.0), precision=mw.MWF_MIXED if c.get("mixed") else mw.MWF_FP64)


def _members(c):
    """(k0, mm, re) of every member of an ensemble; square boxes."""
    ks, ms = [int(x) for x in c["k0"].split(",")], [int(x) for x in c["modes"].split(",")]
    out = []
    for i in range(c["members"]):
        f = (i * 0.618033988749895) % 1.0
        out.append((ks[i % len(ks)], ms[(i // len(ks)) % len(ms)] // 2, c["re"] + c["spread"] * (2 * f - 1)))
    return out


def _classes(c):
    """Members by size: {(k0, mm): [member indices]}."""
    out = {}
    for i, (k0, mm, _) in enumerate(_members(c)):
        out.setdefault((k0, mm), []).append(i)
    return out


class Flow:
    """Model Waleffe Flow in 64 bits from its definition, for a batch of members
    of one size (arrays [member, slot, m or x, n or z])."""

    def __init__(self, c, k0, mm, nn, res):
        self.k0, self.mm, self.nn = k0, mm, nn
        self.K, self.KK, self.M, self.P, self.Q = 2 * k0 - 1, 3 * k0 - 1, 2 * mm - 1, 3 * mm, 3 * nn
        self.dt = c["dt"]
        self.th = c.get("deg", 0.0) / 180.0 * PI
        self.drag = 1e-2
        t = lambda v: torch.as_tensor(v, dtype=F64, device=DEV)  # noqa: E731
        m = np.concatenate([np.arange(mm), np.arange(-(mm - 1), 0)])
        self.rows = t(m % self.P).long()
        self.alpha, self.gamma = 2 * PI / (mm * c["per"]), 2 * PI / (nn * c["per"])
        self.a = t(self.alpha * m)[None, None, :, None]
        self.g = t(self.gamma * np.arange(nn))[None, None, None, :]
        self.ak = t([(-1.0) ** k * k * BETA for k in range(k0)])[None, :, None, None]
        self.re = t(res)[:, None, None, None]

    # mpt <-> spec
    def spec(self, c, lam):
        k0 = self.k0
        psi = c[:, :k0]
        phi = torch.cat([torch.zeros_like(c[:, :1]), c[:, k0:]], 1)
        u = -1j * self.g * psi + 1j * self.a * self.ak * phi
        w = 1j * self.a * psi + 1j * self.g * self.ak * phi
        v = (self.a ** 2 + self.g ** 2) * phi
        u[:, 0, 0, 0] = 0
        w[:, 0, 0, 0] = 0
        u[:, 1:, 0, 0] = psi[:, 1:, 0, 0]
        w[:, 1:, 0, 0] = phi[:, 1:, 0, 0]
        if lam:
            u[:, 1, 0, 0] += math.cos(self.th)
            w[:, 1, 0, 0] += math.sin(self.th)
        return torch.cat([u, v[:, 1:], w], 1)

    def mpt(self, s):
        k0 = self.k0
        u, w = s[:, :k0], s[:, 2 * k0 - 1:]
        v = torch.cat([torch.zeros_like(u[:, :1]), s[:, k0:2 * k0 - 1]], 1)
        psi = -1j * (self.a * w - self.g * u)
        phi = 1j * self.ak * (self.a * u + self.g * w) - (self.a ** 2 + self.g ** 2) * v
        psi[:, 0, 0, 0] = 0
        psi[:, 1:, 0, 0] = -u[:, 1:, 0, 0]
        phi[:, 1:, 0, 0] = -w[:, 1:, 0, 0]
        return torch.cat([psi, phi[:, 1:]], 1)

    # spec <-> phys
    def phys(self, s):
        full = torch.zeros(s.shape[:2] + (self.P, self.nn), dtype=C128, device=DEV)
        full[:, :, self.rows] = s
        f = torch.fft.ifft(full, dim=2, norm="forward")
        f[..., 0].imag.zero_()  # the real transform drops it
        return torch.fft.irfft(f, n=self.Q, dim=3, norm="forward")

    def back(self, p):
        f = torch.fft.rfft(p, dim=3, norm="forward")[..., :self.nn]
        return torch.fft.fft(f.contiguous(), dim=2, norm="forward")[:, :, self.rows]

    def bases(self, y):
        k = np.arange(self.k0)[:, None]
        h = np.where(k % 2 == 0, np.cos(k * BETA * y), np.sin(k * BETA * y))
        g = np.where(k % 2 == 1, np.cos(k * BETA * y), np.sin(k * BETA * y))
        return h, g[1:]

    def products(self):
        """For each pair of families the projection of its products: (row, slot, slot, factor)."""
        y = np.arange(64) / 16.0
        h, g = self.bases(y)
        k0 = self.k0
        sl = {"u": (h, 0), "v": (g, k0), "w": (h, 2 * k0 - 1)}
        out = {}
        for a, b, to in (("u", "u", h), ("u", "w", h), ("w", "w", h), ("u", "v", g), ("v", "w", g), ("v", "v", h)):
            (x, ox), (z, oz) = sl[a], sl[b]
            t = np.einsum("iy,jy,ky->kij", x, z, to) / (to * to).sum(1)[:, None, None]
            out[a + b] = [[(ox + i, oz + j, t[k, i, j]) for i in range(len(x)) for j in range(len(z))
                           if abs(t[k, i, j]) > 1e-9] for k in range(len(to))]
        return out

    def nonlinear(self, c):
        """(u . grad) u = div(u u) of the divergence-free field, as mpt."""
        p, k0 = self.phys(self.spec(c, True)), self.k0
        T = {}
        for name, rows in self.products().items():
            for k, terms in enumerate(rows):
                r = torch.zeros_like(p[:, 0])
                for i, j, f in terms:
                    r.addcmul_(p[:, i], p[:, j], value=f)
                T.setdefault(name, []).append(self.back(r[:, None]))
            T[name] = torch.cat(T[name], 1)
        pad = lambda x: torch.cat([torch.zeros_like(x[:, :1]), x], 1)  # noqa: E731
        ia, ig, ak = 1j * self.a, 1j * self.g, self.ak
        u = ia * T["uu"] + ak * pad(T["uv"]) + ig * T["uw"]
        v = ia * T["uv"] - ak[:, 1:] * T["vv"][:, 1:] + ig * T["vw"]
        w = ia * T["uw"] + ak * pad(T["vw"]) + ig * T["ww"]
        return self.mpt(torch.cat([u, v, w], 1))

    def operators(self):
        dt, k0 = self.dt, self.k0
        hl = -(self.a ** 2) - self.g ** 2
        lap = hl - self.ak ** 2
        tvl = 1.0 - dt * (lap / self.re - self.drag)
        one = torch.ones_like(tvl)
        rp, rq = hl * one, hl * lap * one
        lp, lq = tvl * rp, tvl * rq - dt * self.drag * hl * hl
        for x in (rp, rq):
            x[:, :, 0, 0] = 1.0
        for x in (lp, lq):
            x[:, :, 0, 0] = tvl[:, :, 0, 0]
        rp[:, 0, 0, 0], lp[:, 0, 0, 0] = 0.0, 1.0
        return torch.cat([lp, lq[:, 1:]], 1), torch.cat([rp, rq[:, 1:]], 1)

    def start(self, c):
        self.c, self.old = c, None
        self.lhs, self.rhs = self.operators()

    def step(self, n):
        for _ in range(n):
            nl = self.nonlinear(self.c)
            old = nl if self.old is None else self.old
            self.c = (self.rhs * self.c + self.dt / 2 * (3 * nl - old)) / self.lhs
            self.c[:, 0, 0, 0] = 0
            self.old = nl

    def energy(self, c):
        """Mean square of the perturbation per member (c2r keeps the Hermitian part of n = 0)."""
        s = self.spec(c, False)
        z = s[..., :1]
        z = 0.5 * (z + torch.cat([z[:, :, :1], z[:, :, 1:].flip(2)], 2).conj())
        e = z.abs().square().sum((2, 3)) + 2 * s[..., 1:].abs().square().sum((2, 3))
        y = torch.full((self.KK,), 0.5, dtype=F64, device=DEV)
        y[0] = y[2 * self.k0 - 1] = 1.0
        return (e * y).sum(1)

    def planes(self, c):
        """Re and Im as the framework's arrays: [member, n, m, slot]."""
        return tuple(x.permute(0, 3, 2, 1).contiguous().cpu().numpy() for x in (c.real, c.imag))

    def draw(self, seed, rms, kic):
        """A solenoidal Gaussian-spectrum field of that rms velocity, the laminar mean kept."""
        gen = torch.Generator(device=DEV).manual_seed(seed)
        n = len(self.re)
        c = torch.complex(*(torch.randn((n, self.K, self.M, self.nn), generator=gen, dtype=F64, device=DEV)
                            for _ in range(2)))
        k2 = self.a ** 2 + self.g ** 2
        env = torch.exp(-k2 / kic ** 2) / torch.sqrt(torch.clamp(k2, min=1e-12))
        c[:, :self.k0] *= env
        c[:, self.k0:] *= env / torch.sqrt(k2 + self.ak[:, 1:] ** 2)
        c[:, :, self.mm:, 0] = c[:, :, 1:self.mm, 0].flip(2).conj()
        c[:, :, 0, 0] = 0
        return c * (rms / torch.sqrt(self.energy(c)))[:, None, None, None]

    def eposc(self, p):
        """y means of u^2, v^2, w^2 at the points of phys p: [member, 3, x, z]."""
        k0 = self.k0
        sq = p * p
        return torch.stack([sq[:, 0] + 0.5 * sq[:, 1:k0].sum(1), 0.5 * sq[:, k0:2 * k0 - 1].sum(1),
                            sq[:, 2 * k0 - 1] + 0.5 * sq[:, 2 * k0:].sum(1)], 1)


CT = 1e-2  # turbulent where the local kinetic energy is above 2 % of the laminar one's


def _flow(c, seed):
    f = Flow(c, c["k0"], c["mm"], c["nn"], [c["re"]])
    return f, f.draw(seed, c["rms"], c["k0ic"])


def _ensemble_flows(c, seed):
    mem = _members(c)
    for j, ((k0, mm), idx) in enumerate(_classes(c).items()):
        f = Flow(c, k0, mm, mm, [mem[i][2] for i in idx])
        yield idx, f, f.draw(1000 * seed + j, c["rms"], c["k0ic"])


def prepare(case, seed):
    c = case
    mw.autotune(1 if c["tuned"] else 0)
    try:
        if c["kind"] == "ensemble":
            ens = mw.Ensemble([_params(c, k0, mm, mm, re) for k0, mm, re in _members(c)])
            for idx, f, ic in _ensemble_flows(c, seed):
                re, im = f.planes(ic)
                for k, i in enumerate(idx):
                    ens.set_state(i, re[k], im[k])
            ens.track(c["every"], 1e-6 * 0.5)
            if c["turb"]:
                ens.track_turb(6, 6, CT)
            ens.sync()
            return dict(case=c, ens=ens)
        v = mw.Velocity(_params(c))
    finally:
        mw.autotune(0)
    f, ic = _flow(c, seed)
    re, im = f.planes(ic)
    st = dict(case=c, v=v, re=re[0], im=im[0])
    if c["kind"] == "transform":
        s = f.spec(ic, True)
        p = f.phys(s)
        st["spec"] = tuple(x[0] for x in f.planes(s))
        st["phys"] = (p * p)[0].permute(1, 2, 0).contiguous().cpu().numpy()
    else:
        v.set_state(st["re"], st["im"])
    v.sync()
    return st


# ------------------------------------------------------------------- a pass

def _hand_on(c, x):
    """The mixed form's results go on in single precision, FP64 ones as they are."""
    return torch.from_numpy(x).to(torch.float32) if c.get("mixed") else x


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "ensemble":
        ens = state["ens"]
        ens.step(c["steps"])
        n = c["steps"] // c["every"]
        out = dict(energies=_hand_on(c, ens.energies()))
        if c["steps"] % c["every"] == 0:
            out["trace"] = _hand_on(c, np.stack([ens.trace(i)[0][-n:] for i in range(len(ens))]))
            if c["turb"]:
                out["turb"] = np.stack([ens.trace_turb(i)[-n:] for i in range(len(ens))])
        for j, idx in enumerate(_classes(c).values()):
            re, im = (np.empty((len(idx),) + ens.mpt_shape(idx[0])) for _ in range(2))
            for k, i in enumerate(idx):
                re[k], im[k] = ens.get_state(i)
            out["re%d" % j], out["im%d" % j] = _hand_on(c, re), _hand_on(c, im)
        return out
    v = state["v"]
    if kind == "run":
        e = np.empty(c["blocks"])
        for b in range(c["blocks"]):
            v.vel_TS(c["every"])
            e[b] = v.vel_energy()
        re, im = v.get_state()
        return dict(energy=_hand_on(c, e), re=_hand_on(c, re), im=_hand_on(c, im))
    if kind == "monitor":
        v.vel_TS(c["steps"])
        e = v.vel_energy()
        m_max, n_max = v.spectrum_max()
        return dict(energy=e, m_max=m_max, n_max=n_max, history=v.vel_history(8, 0.25),
                    turb=v.turb_sample(c["stride"], c["stride"]), fraction=v.turb_fraction(6, 6, CT))
    if kind == "field":
        re, im = v.vel_nonlinear()
        ph = v.vel_mpt2phys(state["re"], state["im"])
        return dict(re=_hand_on(c, re), im=_hand_on(c, im), phys=_hand_on(c, ph))
    ph = v.tra_spec2phys(*state["spec"])
    re, im = v.tra_phys2spec(state["phys"])
    return dict(phys=_hand_on(c, ph), re=_hand_on(c, re), im=_hand_on(c, im))


# -------------------------------------------------------------------- the work

def _step_work(k0, mm, nn, mixed):
    """Bytes and operations of one step: state and history read and written, and
    the velocity taken to the grid and the products back, through x-physical
    z-spectral arrays that no on-chip memory holds, written and read once each."""
    K, KK, M, P, Q, s = 2 * k0 - 1, 3 * k0 - 1, 2 * mm - 1, 3 * mm, 3 * nn, 8 if mixed else 16
    b = (2 * 16 + 2 * s) * K * M * nn + 4 * s * KK * P * nn
    f = 2 * KK * (5 * P * math.log2(P) * nn + 2.5 * Q * math.log2(Q) * P) + 2 * P * Q * 5 * KK
    return b, f


def work(case):
    c = case
    if c["kind"] == "ensemble":
        b = f = 0.0
        for k0, mm, _ in _members(c):
            x, y = _step_work(k0, mm, mm, c["mixed"])
            b += c["steps"] * x + 2 * 16 * (2 * k0 - 1) * (2 * mm - 1) * mm
            f += c["steps"] * y
        return dict(bytes=b, flops=f)
    k0, mm, nn = c["k0"], c["mm"], c["nn"]
    K, KK, M, P, Q = 2 * k0 - 1, 3 * k0 - 1, 2 * mm - 1, 3 * mm, 3 * nn
    b, f = _step_work(k0, mm, nn, c.get("mixed"))
    st, ph = 16 * K * M * nn, 8 * KK * P * Q
    s = 8 if c.get("mixed") else 16
    half = KK * (5 * P * math.log2(P) * nn + 2.5 * Q * math.log2(Q) * P)
    if c["kind"] == "run":
        n = c["every"] * c["blocks"]
        return dict(bytes=n * b + (c["blocks"] + 2) * st, flops=n * f)
    if c["kind"] == "monitor":
        line = 2 * s * KK * P * nn
        return dict(bytes=c["steps"] * b + 3 * st + line + 2 * ph, flops=c["steps"] * f + half)
    if c["kind"] == "field":
        return dict(bytes=4 * st + 6 * s * KK * P * nn + ph, flops=f + half)
    return dict(bytes=2 * 16 * KK * M * nn + 4 * s * KK * P * nn + 2 * ph, flops=2 * half)


# ---------------------------------------------------------------- in 64 bits

def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "ensemble":
        n = c["steps"] // c["every"]
        out, e = {}, np.empty(c["members"])
        tr, tu = np.empty((c["members"], n)), np.empty((c["members"], n))
        for j, (idx, f, ic) in enumerate(_ensemble_flows(c, seed)):
            f.start(ic)
            for b in range(n):
                f.step(c["every"])
                tr[idx, b] = f.energy(f.c).cpu().numpy()
                if c["turb"]:
                    ep = f.eposc(f.phys(f.spec(f.c, False)))[:, :, ::6, ::6].sum(1)
                    tu[idx, b] = ((ep > CT).sum((1, 2)).double() / ((f.Q // 6 + 1.0) * (f.P // 6 + 1))).cpu().numpy()
            f.step(c["steps"] - n * c["every"])
            e[idx] = f.energy(f.c).cpu().numpy()
            out["re%d" % j], out["im%d" % j] = f.planes(f.c)
        out["energies"] = e
        if c["steps"] % c["every"] == 0:
            out["trace"] = tr
            if c["turb"]:
                out["turb"] = tu
        return out
    f, ic = _flow(c, seed)
    if kind == "run":
        f.start(ic)
        e = np.empty(c["blocks"])
        for b in range(c["blocks"]):
            f.step(c["every"])
            e[b] = float(f.energy(f.c)[0])
        re, im = f.planes(f.c)
        return dict(energy=e, re=re[0], im=im[0])
    if kind == "monitor":
        f.start(ic)
        f.step(c["steps"])
        s = f.spec(f.c, False)
        p = f.phys(s)
        d = s.abs()[0].amax(0)
        m_max = d.amax(1)
        m_max = torch.maximum(m_max[:f.mm], torch.cat([m_max[:1], m_max[f.mm:].flip(0)]))
        ep = f.eposc(p)[0]
        frac = float((ep.sum(0)[::6, ::6] > CT).sum()) / ((f.Q // 6 + 1.0) * (f.P // 6 + 1))
        h, g = (torch.as_tensor(x, device=DEV) for x in f.bases(0.25))
        ji = torch.as_tensor([(j * f.Q) // 8 + 1 for j in range(8)], device=DEV)
        at, k0 = p[0, :, 0][:, ji], c["k0"]
        hist = torch.stack([ji.double() * (c["nn"] * c["per"]) / f.Q, (h * at[:k0]).sum(0), (g * at[k0:2 * k0 - 1]).sum(0),
                            (h * at[2 * k0 - 1:]).sum(0)], 1)
        q = c["stride"]
        sm, sn = f.P // q, f.Q // q
        t = ep[:, :sm * q:q, :sn * q:q].permute(1, 2, 0)
        return dict(energy=float(f.energy(f.c)[0]), m_max=m_max.cpu().numpy(), n_max=d.amax(0).cpu().numpy(),
                    history=hist.cpu().numpy(), turb=t.contiguous().cpu().numpy(), fraction=frac)
    if kind == "field":
        re, im = f.planes(f.nonlinear(ic))
        p = f.phys(f.spec(ic, False))[0].permute(1, 2, 0).contiguous().cpu().numpy()
        return dict(re=re[0], im=im[0], phys=p)
    s = f.spec(ic, True)
    p = f.phys(s)
    re, im = f.planes(f.back(p * p))
    return dict(phys=p[0].permute(1, 2, 0).contiguous().cpu().numpy(), re=re[0], im=im[0])
