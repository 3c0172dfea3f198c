"""Performance cases: the work a user of ps3d_amd has it do, through the package's
public entry points (ps3d_amd.gpu, ps3d_amd.closure).

Kinds of case
  advance   ps3d's production run: `steps` time steps of one grid, then the state to
            the host, as a run does between two output times.
  until     the host program's loop (`do while t < limit`) on a small grid: up to nmax
            gated steps to the next output time.
  ensemble  batched groups of small grids stepped together, then their states.
  output    an output time: inversion, adapt, pressure and divergence, the field_stats
            record, genspec's spectrum, and the physical fields to the host.
  operator  single horizontal transforms on host arrays.
  train     loss and gradients of the learned closure on one sample.
  coupled   a coarse run with the trained closure attached.

Grid lengths are even numbers 2^a 3^b 5^c, the lengths the framework takes; the flows
are its benchmark's (Beltrami modes with noise, random-phase isotropic turbulence made on
the grid itself or on a coarser one and zero-padded).
"""
import math
import os

import numpy as np
import torch

from ps3d_amd import closure as CL
from ps3d_amd import closure_run as CR
from ps3d_amd import gpu as G

PI = math.pi
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "ps3d_amd", "data", "closure64.npz")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _advance(nx, ny, nz, steps, ic, filtering="2/3-rule", stepper="impl-diff-rk4", pretype="vorch"):
    return dict(kind="advance", nx=nx, ny=ny, nz=nz, steps=steps, ic=ic, filtering=filtering, stepper=stepper,
                pretype=pretype)


def listed():
    return [
        # the smallest calls: one operator on a host array, where copies and launches are all
        dict(kind="operator", nx=32, ny=32, nz=32, name="operator-32"),
        # the validation run (fixed step 0.01) as the host program drives it to its next output
        dict(kind="until", nx=32, ny=32, nz=32, steps=20, name="until-32"),
        # ordinary run: 128^3, adaptive step
        dict(_advance(128, 128, 128, 30, "beltrami"), name="advance-128"),
        # the headline benchmark's grid and flow
        dict(_advance(256, 256, 256, 20, "beltrami"), name="advance-256"),
        # the largest: turbulence spun up on 128^3 and zero-padded to 512^3
        dict(_advance(512, 512, 512, 8, "padded"), name="advance-512"),
        # ps3d's default options (Hou & Li filter, rolling-mean prefactor) on a grid with
        # three different lengths, none of them a power of two
        dict(_advance(160, 90, 100, 20, "random", "Hou & Li", "impl-diff-rk4", "roll-mean-max-strain"),
             name="advance-160x90x100"),
        # the other time stepper
        dict(_advance(96, 96, 96, 20, "random", "2/3-rule", "cn2", "vorch"), name="cn2-96"),
        # an uneven ensemble in the benchmark's proportions (40/30/20/10 %)
        dict(kind="ensemble", n32=12, n48=9, n64=6, n96=3, steps=20, name="ensemble-30"),
        # one output time of the 128^3 run
        dict(kind="output", nx=128, ny=128, nz=128, name="output-128"),
        # one training sample of the 64^3 closure
        dict(kind="train", n=64, name="closure-train-64"),
        # the coarse run the closure was trained for
        dict(kind="coupled", n=64, steps=40, name="closure-run-64"),
    ]


def _length(rng, lo, hi):
    """An even 2^a 3^b 5^c between lo and hi, spread over the logarithm."""
    while True:
        n = 2 * round(math.exp(rng.uniform(math.log(lo / 2), math.log(hi / 2))))
        if _smooth(n) and lo <= n <= hi:
            return n


def draw(rng):
    kind = rng.choice(["advance"] * 5 + ["until", "ensemble", "output", "operator", "train"])
    if kind == "ensemble":
        return dict(kind=kind, n32=rng.randint(1, 24), n48=rng.randint(1, 16), n64=rng.randint(1, 10),
                    n96=rng.randint(0, 5), steps=rng.randint(5, 25))
    if kind == "train":
        return dict(kind=kind, n=_length(rng, 32, 80))
    if kind in ("output", "operator", "until"):
        hi = 64 if kind == "until" else 160
        c = dict(kind=kind, nx=_length(rng, 24, hi), ny=_length(rng, 24, hi), nz=_length(rng, 24, hi))
        if kind == "until":
            c["steps"] = rng.randint(5, 40)
        return c
    if rng.random() < 0.5:   # cubes, as most runs are
        nx = ny = nz = _length(rng, 24, 384)
    else:
        nx, ny, nz = (_length(rng, 24, 384) for _ in range(3))
    most = max(2, min(40, int(8 * 512 ** 3 / (nx * ny * nz * 8.0))))
    return _advance(nx, ny, nz, rng.randint(2, most), rng.choice(["beltrami", "random", "padded"]),
                    rng.choice(["2/3-rule", "2/3-rule", "Hou & Li"]),
                    rng.choice(["impl-diff-rk4", "impl-diff-rk4", "impl-diff-rk4", "cn2"]),
                    rng.choice(["vorch", "roll-mean-max-strain"]))


# ---------------------------------------------------------------------------
# initial flows (on the GPU, from the seed)
# ---------------------------------------------------------------------------
BOX = (2 * PI, 2 * PI, PI)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _beltrami(nx, ny, nz, seed):
    """Vorticity of four Beltrami modes with random phases plus 1e-3 noise."""
    g = _gen(seed)
    f8 = dict(dtype=torch.float64, device="cuda")
    x = torch.arange(nx, **f8).view(-1, 1, 1) * (BOX[0] / nx)
    y = torch.arange(ny, **f8).view(1, -1, 1) * (BOX[1] / ny)
    z = torch.arange(nz + 1, **f8).view(1, 1, -1) * (BOX[2] / nz)
    phase = torch.rand(4, generator=g, **f8) * (2 * PI)
    vor = 1e-3 * torch.randn(3, nx, ny, nz + 1, generator=g, **f8)
    for (k, l, m), ph in zip(((1, 1, 1), (2, 1, 1), (1, 2, 1), (2, 2, 2)), phase):
        a = math.sqrt(k * k + l * l + m * m)
        sm, cm = torch.sin(m * z), torch.cos(m * z)
        th = k * x + l * y + ph
        s, c = torch.sin(th), torch.cos(th)
        f = a / (k * k + l * l)
        vor[0] += f * (-k * m * cm - l * a * sm) * s
        vor[1] += f * (-l * m * cm + k * a * sm) * s
        vor[2] += a * sm * c
    return vor


def _random(nx, ny, nz, seed, k0=4.0):
    """Vorticity of a solenoidal random-phase flow, E(k) ~ k^4 exp(-2 (k/k0)^2), unit
    rms speed, w = 0 on the lids: the curl of a potential with sine (x, y components)
    and cosine (z component) series in z."""
    g = _gen(seed)
    f8 = dict(dtype=torch.float64, device="cuda")
    kx = (torch.fft.fftfreq(nx, d=1.0 / nx, **f8) * (2 * PI / BOX[0])).view(-1, 1, 1)
    ky = (torch.fft.fftfreq(ny, d=1.0 / ny, **f8) * (2 * PI / BOX[1])).view(1, -1, 1)
    mz = (torch.arange(nz + 1, **f8) * (PI / BOX[2])).view(1, 1, -1)
    K2 = kx ** 2 + ky ** 2 + mz ** 2
    amp = torch.exp(-K2 / k0 ** 2) * (K2 > 0) * (kx.abs() <= 2 / 3 * kx.abs().max()) \
        * (ky.abs() <= 2 / 3 * ky.abs().max()) * (mz <= 2 / 3 * mz.max())
    A = [amp * torch.complex(torch.randn(K2.shape, generator=g, **f8), torch.randn(K2.shape, generator=g, **f8))
         for _ in range(3)]
    ang = torch.outer(mz.flatten(), torch.arange(nz + 1, **f8) * (BOX[2] / nz))
    S, C = torch.sin(ang).to(torch.complex128), torch.cos(ang).to(torch.complex128)

    def synth(coef, basis):
        return torch.fft.ifft2(coef @ basis, dim=(0, 1)).real * (nx * ny)

    U = 1j * ky * A[2] - mz * A[1]
    V = mz * A[0] - 1j * kx * A[2]
    W = 1j * kx * A[1] - 1j * ky * A[0]
    rms = torch.sqrt(sum(synth(c, b).square().mean() for c, b in ((U, C), (V, C), (W, S))) / 3)
    return torch.stack([synth(1j * ky * W + mz * V, S), synth(-mz * U - 1j * kx * W, S),
                        synth(1j * kx * V - 1j * ky * U, C)]) / rms


def _coarse(n):
    """The grid a padded flow is made on: a half to a quarter of the length, at most 128."""
    m = min(128, max(16, n // 2))
    while not _smooth(m):
        m -= 1
    return m


def _smooth(n):
    """An even 2^a 3^b 5^c."""
    m = n
    for p in (2, 3, 5):
        while m % p == 0:
            m //= p
    return m == 1 and n % 2 == 0


def _initial(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ic = case.get("ic", "beltrami")
    if ic == "padded":
        return _random(_coarse(nx), _coarse(ny), _coarse(nz), seed)
    return (_random if ic == "random" else _beltrami)(nx, ny, nz, seed)


def _params(nx, ny, nz, case):
    return G.make_params(nx, ny, nz, lower=(0.0, 0.0, 0.0), extent=BOX,
                         filtering=case.get("filtering", "2/3-rule"), stepper=case.get("stepper", "impl-diff-rk4"),
                         nnu=3, prediss=30.0, pretype=case.get("pretype", "vorch"), roll_mean_win_size=1000,
                         length_scale="Kolmogorov", alpha=0.1, limit=1.0e30,
                         dt_fixed=0.01 if case["kind"] == "until" else 0.0)


def _solver(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = G.Ps3dGpu(_params(nx, ny, nz, case))
    vor = _initial(case, seed).cpu().numpy()
    if case.get("ic") == "padded":
        src = G.Ps3dGpu(_params(_coarse(nx), _coarse(ny), _coarse(nz), case))
        src.set_vorticity(vor)
        G.resample(h, src)
        src.close()
    else:
        h.set_vorticity(vor)
    return h


def _members(case):
    return [(n, case["n%d" % n]) for n in (32, 48, 64, 96) if case["n%d" % n]]


def _sample(n, seed):
    """One training sample: the six smooth input fields of unit variance, and a target."""
    g = _gen(seed)
    x = torch.randn(n * n * (n + 1), 6, generator=g, device="cuda")
    t = torch.randn(n * n * (n + 1), 3, generator=g, device="cuda")
    return x, t


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("advance", "until", "output"):
        return dict(kind=kind, case=case, h=_solver(case, seed))
    if kind == "operator":
        h = G.Ps3dGpu(_params(case["nx"], case["ny"], case["nz"], case))
        return dict(kind=kind, h=h, f=_beltrami(case["nx"], case["ny"], case["nz"], seed)[0].cpu().numpy())
    if kind == "ensemble":
        mem = _members(case)
        ens = G.Ps3dEnsemble([_params(n, n, n, case) for n, _ in mem], [c for _, c in mem])
        k0 = np.random.default_rng(seed).uniform(2.0, 6.0, size=sum(c for _, c in mem))
        i = 0
        for grp, (n, c) in zip(ens.groups, mem):
            for b in range(c):
                grp.set_vorticity(b, _random(n, n, n, seed + i, float(k0[i])).cpu().numpy())
                i += 1
        return dict(kind=kind, case=case, ens=ens)
    if kind == "train":
        n = case["n"]
        net = CL.ClosureNet(n, n, n)
        net.set_weights(CL.init_weights(7))
        x, t = _sample(n, seed)
        return dict(kind=kind, net=net, x=x.cpu().numpy(), t=t.cpu().numpy())
    net, gain, prediss, _ = CR.load_net(WEIGHTS, case["n"])   # coupled
    net.out_scale = net.out_scale * gain
    h = G.Ps3dGpu(CR.params(case["n"], prediss=prediss))
    h.set_vorticity(_random(case["n"], case["n"], case["n"], seed, 5.0).cpu().numpy())
    net.attach(h)
    return dict(kind=kind, case=case, h=h, net=net)


def run(state):
    kind = state["kind"]
    if kind in ("advance", "coupled"):
        h = state["h"]
        return {"diag": h.advance_n(state["case"]["steps"]), "svor": h.get(G.SVOR)}
    if kind == "until":
        h, n = state["h"], state["case"]["steps"]
        # the output time lies between two steps; the loop has room for a few more
        return {"diag": h.advance_until(h.t + 0.01 * n - 0.005, n + 5), "svor": h.get(G.SVOR)}
    if kind == "output":
        h = state["h"]
        h.vor2vel()
        dt, diag = h.adapt(h.t)
        h.derived()
        stats = h.field_stats(diag)
        out = {"dt": dt, "diag": diag, "stats": stats, "vel": h.get(G.VEL), "vor": h.get(G.VOR),
               "pres": h.get(G.PRES), "delta": h.get(G.DELTA)}
        k, spec, num = h.spectrum()
        out.update(spec=spec, num=num)
        return out
    if kind == "operator":
        fs = state["h"].fftxyp2s(state["f"])
        return {"fs": fs, "fz": state["h"].fftxys2p(state["h"].central_diffz(fs))}
    if kind == "ensemble":
        ens = state["ens"]
        ens.advance(state["case"]["steps"])
        return {"n%d" % g.shape[0]: np.stack([g.get_svor(b) for b in range(g.nbatch)]) for g in ens.groups}
    loss, g, gx = state["net"].grad(state["x"], state["t"], want_gx=True)   # train
    return {"loss": loss, "grad": g, "gx": gx}


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def _step_work(nx, ny, nz, stages):
    """One time step: each volume a pass cannot keep on chip, once in and once out.  A
    stage writes and reads six fields between the z and y and between the y and x
    passes, three back, and about eight more in the update; the adapt stage three
    derivative fields through y and x and the six fields it evaluates."""
    n = nx * ny * (nz + 1)
    vol = 36 * stages + 8 * stages + 15
    lg = 2.5 * math.log2(nx * ny)
    flops = n * (stages * (9 * lg + 12 * 2.5 * math.log2(2 * nz) + 60) + 6 * lg + 60)
    return 8.0 * n * vol, flops


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        b = f = 0.0
        for n, c in _members(case):
            w = _step_work(n, n, n, 4)
            b += c * (case["steps"] * w[0] + 6 * 8.0 * n * n * (n + 1))
            f += c * case["steps"] * w[1]
        return {"bytes": b, "flops": f}
    if kind == "train":
        n = case["n"] ** 2 * (case["n"] + 1)
        return {"bytes": n * 4.0 * (6 + 3 + 6), "flops": 3e9 * CL.GFLOP_FWD_PER_POINT * n}
    if kind == "coupled":
        n, s = case["n"], case["steps"]
        w, npts = _step_work(n, n, n, 4), n * n * (n + 1)
        return {"bytes": s * w[0] + 48.0 * npts, "flops": s * (w[1] + 1e9 * CL.GFLOP_FWD_PER_POINT * npts)}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * (nz + 1)
    lg = 2.5 * math.log2(nx * ny)
    if kind == "operator":
        return {"bytes": 6 * 8.0 * n, "flops": n * (2 * lg + 2)}
    if kind == "output":
        return {"bytes": 8.0 * n * (3 + 8), "flops": n * (16 * lg + 14 * 2.5 * math.log2(2 * nz) + 200)}
    w = _step_work(nx, ny, nz, 3 if case.get("stepper") == "cn2" else 4)
    return {"bytes": case["steps"] * w[0] + 6 * 8.0 * n, "flops": case["steps"] * w[1]}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _pack(f, dim):
    """Unitary real transform in Hermitian order: cosine parts 0..n/2, then sine parts."""
    n = f.shape[dim]
    a = torch.fft.rfft(f, dim=dim, norm="ortho")
    return torch.cat([a.real, a.imag.narrow(dim, 1, n // 2 - 1).flip(dim)], dim)


def _unpack(s, dim):
    n = s.shape[dim]
    re = s.narrow(dim, 0, n // 2 + 1)
    im = torch.zeros_like(re)
    im.narrow(dim, 1, n // 2 - 1).copy_(s.narrow(dim, n // 2 + 1, n // 2 - 1).flip(dim))
    return torch.fft.irfft(torch.complex(re, im), n=n, dim=dim, norm="ortho")


def _p2s(f):
    return _pack(_pack(f, -2), -3)


def _s2p(s):
    return _unpack(_unpack(s, -3), -2)


def _sine(f):
    """DST-I of the interior levels; the lids stay."""
    nz = f.shape[-1] - 1
    ext = torch.cat([torch.zeros_like(f[..., :1]), f[..., 1:nz], torch.zeros_like(f[..., :1]), -f[..., 1:nz].flip(-1)], -1)
    s = -torch.fft.rfft(ext).imag[..., 1:nz] / math.sqrt(2.0 * nz)
    return torch.cat([f[..., :1], s, f[..., nz:]], -1)


def _cosine(f):
    nz = f.shape[-1] - 1
    return torch.fft.rfft(torch.cat([f, f[..., 1:nz].flip(-1)], -1)).real / math.sqrt(2.0 * nz)


class _Exact:
    """The time step's mathematics: packed horizontal spectra at the z levels."""

    def __init__(self, nx, ny, nz, case, dt_fixed=0.0):
        f8 = dict(dtype=torch.float64, device="cuda")
        self.n, self.dt_fixed = (nx, ny, nz), dt_fixed
        self.hou = case.get("filtering") == "Hou & Li"
        self.cn2, self.pretype = case.get("stepper") == "cn2", case.get("pretype", "vorch")
        k = [torch.minimum(torch.arange(n, **f8), n - torch.arange(n, **f8)) * (2 * PI / L)
             for n, L in ((nx, BOX[0]), (ny, BOX[1]))]
        kz = torch.arange(nz + 1, **f8) * (PI / BOX[2])
        self.kz = kz
        self.f = []
        for kk, n in zip(k, (nx, ny)):   # derivative factor of slot j on slot n - j
            w = torch.where(torch.arange(n, device="cuda") > n // 2, kk, -kk)
            w[0] = w[n // 2] = 0.0
            self.f.append(w)
        self.f[0], self.f[1] = self.f[0].view(-1, 1, 1), self.f[1].view(1, -1, 1)
        self.k2 = (k[0].view(-1, 1) ** 2 + k[1].view(1, -1) ** 2).unsqueeze(-1)
        self.k2i = torch.where(self.k2 > 0, 1.0 / self.k2, torch.zeros_like(self.k2))
        self.k2max = max(float(k[0].max()), float(k[1].max())) ** 2
        if self.hou:
            e = [-36.0 * (kk / kk.max()) ** 36 for kk in (*k, kz)]
            self.f0 = torch.exp(e[0].view(-1, 1, 1) + e[1].view(1, -1, 1))
            self.fz = torch.exp(e[2])
        else:
            m = [(kk <= (2.0 / 3.0) * kk.max()).to(torch.float64) for kk in (*k, kz)]
            self.f0 = m[0].view(-1, 1, 1) * m[1].view(1, -1, 1)
            self.fz = m[2]
        self.f0[0, 0] = 1.0
        self.fz[0] = self.fz[-1] = 1.0
        self.dz = BOX[2] / nz
        zp = torch.arange(nz + 1, **f8) * self.dz
        zm = BOX[2] - zp
        K, Lz = torch.sqrt(self.k2), BOX[2]
        ef = torch.exp(-K * Lz)
        with_k = self.k2 > 0
        div = torch.where(with_k, 1.0 / (1.0 - ef * ef), torch.zeros_like(ef))
        ep, em = torch.exp(-K * zp), torch.exp(-K * zm)
        self.pm = torch.where(with_k, div * (ep - ef * em), (zm / Lz).expand_as(ep))
        self.pp = torch.where(with_k, div * (em - ef * ep), (zp / Lz).expand_as(ep))
        dm, dp = -K * div * (ep + ef * em), K * div * (em + ef * ep)
        Q, R, h, Lm, Lp = div * (1 + ef * ef), div * 2 * ef, 0.5 * self.k2i, K * zm, K * zp
        self.tm = h * (R * Lm * self.pp - Q * Lp * self.pm)
        self.tp = h * (R * Lp * self.pm - Q * Lm * self.pp)
        self.dtm = -h * ((Q * Lp - 1) * dm - R * Lm * dp)
        self.dtp = -h * ((Q * Lm - 1) * dp - R * Lp * dm)
        self.gt = 0.5 * Lz * ((zp / Lz) ** 2 - 1.0 / 3.0)
        self.hist = []

    def dx(self, s):
        return self.f[0] * s.flip(-3).roll(1, -3)

    def dy(self, s):
        return self.f[1] * s.flip(-2).roll(1, -2)

    def dzc(self, s):
        d = torch.empty_like(s)
        d[..., 1:-1] = (s[..., 2:] - s[..., :-2]) * (0.5 / self.dz)
        d[..., 0] = (s[..., 1] - s[..., 0]) / self.dz
        d[..., -1] = (s[..., -1] - s[..., -2]) / self.dz
        return d

    def decompose(self, s, at=slice(None)):
        """Semi-spectral -> mixed: harmonic part of the lid values off, sine series."""
        t = s - (s[..., :1] * self.pm[at] + s[..., -1:] * self.pp[at])
        t[..., 0], t[..., -1] = s[..., 0], s[..., -1]
        return _sine(t)

    def combine(self, s):
        t = _sine(s) + (s[..., :1] * self.pm + s[..., -1:] * self.pp)
        t[..., 0], t[..., -1] = s[..., 0], s[..., -1]
        return t

    def invert(self, q):
        """Projection and velocity of semi-spectral vorticity q (3, ...): (q, u)."""
        d = self.dx(q[1]) - self.dy(q[0])
        e = self.dzc(q[2])
        a = self.k2i * (self.dx(e) + self.dy(d))
        b = self.k2i * (self.dy(e) - self.dx(d))
        a[0, 0], b[0, 0] = q[0][0, 0], q[1][0, 0]
        ds = self.decompose(self.dy(a) - self.dx(b))
        d0, dn = ds[..., :1], ds[..., -1:]
        bs, es = d0 * self.tm + dn * self.tp, d0 * self.dtm + dn * self.dtp
        ds = -ds / (self.k2 + self.kz ** 2).clamp(min=1e-300)
        ds[..., 0] = ds[..., -1] = 0.0
        es = es + _cosine(self.kz * ds)
        w = _sine(ds) + bs
        w[..., 0] = w[..., -1] = 0.0
        u = self.k2i * (self.dx(es) + self.dy(q[2]))
        v = self.k2i * (self.dy(es) - self.dx(q[2]))
        kzi = 1.0 / self.kz.clamp(min=1e-300)
        kzi[0] = kzi[-1] = 0.0
        A, B = self.decompose(torch.stack([a[0, 0], b[0, 0]]), (0, 0))
        u[0, 0] = _cosine(-kzi * B) + B[-1] * self.gt - B[0] * self.gt.flip(0)
        v[0, 0] = _cosine(kzi * A) - A[-1] * self.gt + A[0] * self.gt.flip(0)
        return torch.stack([a, b, q[2]]), torch.stack([u, v, w])

    def source(self, up, op):
        r = _p2s(up[0] * op[1] - up[1] * op[0])
        q = _p2s(up[2] * op[0] - up[0] * op[2])
        p = _p2s(up[1] * op[2] - up[2] * op[1])
        return torch.stack([self.dy(r) - self.dzc(q), self.dzc(p) - self.dx(r), self.dx(q) - self.dy(p)])

    def mean(self, f):
        m = f.sum((-3, -2))
        m = m[..., 1:-1].sum(-1) + 0.5 * (m[..., 0] + m[..., -1])
        return m / (self.n[0] * self.n[1] * self.n[2])

    def start(self, q):
        q, u = self.invert(q)
        ke, en = (0.5 * float(self.mean((_s2p(f) ** 2).sum(0))) for f in (u, q))
        self.visc = 30.0 * (self.k2max * ke / en) ** (1.0 / 3.0) / self.k2max ** 3
        self.ini = [self.barmean(q[c]) for c in (0, 1)]
        return q

    def barmean(self, s):
        c = s[0, 0] / math.sqrt(self.n[0] * self.n[1])
        return float(c[1:-1].sum() + 0.5 * (c[0] + c[-1])) / self.n[2]

    def adapt(self, t, u, up, op):
        eps = 1e-12
        w2 = (op ** 2).sum(0)
        rms = math.sqrt(float(self.mean(w2)))
        mid = (0.5 * (op[..., 1:] + op[..., :-1])).abs()
        l1, l2 = mid.sum(0), (mid ** 2).sum(0)
        on = l1 > rms
        vorch = float((l2 * on).sum() / (eps + (l1 * on).sum()))
        a, c = _s2p(self.dx(u[0])), _s2p(self.dy(u[1]))
        b = _s2p(self.dy(u[0])) + 0.5 * op[2]
        d = _s2p(self.dx(u[2])) + 0.5 * op[1]
        e = _s2p(self.dy(u[2])) - 0.5 * op[0]
        # largest |eigenvalue| of the traceless strain, from its characteristic cubic
        g = -(a + c)
        p = torch.sqrt(((a * a + c * c + g * g) + 2 * (b * b + d * d + e * e)) / 6.0).clamp(min=1e-300)
        det = a * (c * g - e * e) - b * (b * g - e * d) + d * (b * e - c * d)
        th = torch.acos((0.5 * det.abs() / p ** 3).clamp(max=1.0)) / 3.0
        lam = 2.0 * p * torch.cos(th)
        gg, us, ls = float(lam.max()), float(lam[..., -1].max()), float(lam[..., 0].max())
        mx = [float(f.max()) for f in up]
        h = [BOX[i] / self.n[i] for i in range(3)]
        dt = min(0.1 / (gg + eps), 0.1 / eps, 0.8 * min(h[i] / (mx[i] + eps) for i in range(3)), 1e30 - t)
        if self.dt_fixed:
            dt = min(self.dt_fixed, 1e30 - t)
        self.hist.append(gg)
        rg = sum(self.hist[-1000:]) / min(1000, len(self.hist))
        pref = {"vorch": vorch, "roll-mean-max-strain": rg}[self.pretype]
        mean = [self.barmean(_p2s(op[i])) for i in range(3)]
        diag = [t, dt, 0.5 * float(self.mean((up ** 2).sum(0))), 0.5 * float(self.mean(w2)),
                float(self.mean((up * op).sum(0))), math.sqrt(float(w2.max())), rms, vorch, *mean, gg, *mx, us, ls, rg,
                pref]
        return dt, pref, diag

    def restore(self, q):
        for c in (0, 1):
            q[c][0, 0] += (self.ini[c] - self.barmean(q[c])) * math.sqrt(self.n[0] * self.n[1])
        return q

    def filtered(self, q):
        """All three filter factors, the vertical one on the sine coefficients."""
        fz = self.fz.expand(*self.f0.shape[:2], -1).clone()
        fz[0, 0] = 1.0
        return self.combine(self.f0 * fz * self.decompose(q))

    def step(self, t, q):
        q, u = self.invert(q)
        up, op = _s2p(u), _s2p(q)
        dt, pref, diag = self.adapt(t, u, up, op)
        s = self.source(up, op)
        rate = self.visc * self.k2 ** 3
        if self.cn2:
            damp = 1.0 / (1.0 + pref * dt * rate)
            q0 = q + 0.5 * dt * s
            for it in range(3):
                if it:
                    q, u = self.invert(q)
                    s = self.source(_s2p(u), _s2p(q))
                q = self.restore(damp * self.filtered(q0 + 0.5 * dt * s))
            return t + dt, q, diag
        D = 0.5 * pref * dt * rate
        em, ep = torch.exp(-D), torch.exp(D)
        k = [self.f0 * s]
        for c, w in ((0.5, em), (0.5, em), (1.0, em * em)):
            g = (self.f0, ep * self.f0, ep * self.f0)[len(k) - 1]
            qs, u = self.invert(w * (q + c * dt * k[-1]))
            s = self.source(_s2p(u), _s2p(qs))
            k.append((ep * self.f0 if len(k) < 3 else (ep * self.f0) ** 2) * s)
        q = em * em * (q + dt * (k[0] / 6 + k[1] / 3 + k[2] / 3 + k[3] / 6))
        return t + dt, self.restore(q), diag

    def run(self, q, steps):
        t, rows = 0.0, []
        for _ in range(steps):
            t, q, d = self.step(t, q)
            rows.append(d)
        return np.array(rows), self.decompose(q)


def _exact_net(case, seed):
    """The closure's loss and gradients by plain matrix products."""
    n = case["n"]
    x, t = (a.double() for a in _sample(n, seed))
    x = x.requires_grad_(True)
    flat = torch.tensor(CL.init_weights(7), dtype=torch.float64, device="cuda", requires_grad=True)
    a, at = x.view(n, n, n + 1, 6), 0
    for i, (ci, co) in enumerate(CL.LAYERS):
        W, at = flat[at:at + 27 * ci * co].view(27, co, ci), at + 27 * ci * co
        b, at = flat[at:at + co], at + co
        pad = torch.nn.functional.pad(a, (0, 0, 1, 1))
        y = b.expand(n, n, n + 1, co)
        for tap in range(27):
            ox, oy, oz = tap // 9 - 1, tap // 3 % 3 - 1, tap % 3
            y = y + torch.roll(pad[:, :, oz:oz + n + 1], (-ox, -oy), (0, 1)) @ W[tap].T
        a = torch.nn.functional.gelu(y) if i < 3 else y
    loss = (a.reshape(-1, 3) - t).square().mean()
    loss.backward()
    return {"loss": float(loss), "grad": flat.grad, "gx": x.grad}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_net(case, seed)
    if kind == "coupled":
        return None
    if kind == "ensemble":
        k0 = np.random.default_rng(seed).uniform(2.0, 6.0, size=sum(c for _, c in _members(case)))
        out, i = {}, 0
        for n, c in _members(case):
            got = []
            for _ in range(c):
                e = _Exact(n, n, n, case)
                got.append(e.run(e.start(_p2s(_random(n, n, n, seed + i, float(k0[i])))), case["steps"])[1])
                i += 1
            out["n%d" % n] = torch.stack(got)
        return out
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if nx * ny * nz > 300 ** 3 or case.get("ic") == "padded":
        return None
    if kind == "operator":
        e = _Exact(nx, ny, nz, case)
        fs = _p2s(_beltrami(nx, ny, nz, seed)[0])
        return {"fs": fs, "fz": _s2p(e.dzc(fs))}
    e = _Exact(nx, ny, nz, case, 0.01 if kind == "until" else 0.0)
    q = e.start(_p2s(_initial(case, seed)))
    if kind == "output":
        q, u = e.invert(q)
        up, op = _s2p(u), _s2p(q)
        dt, _, diag = e.adapt(0.0, u, up, op)
        return {"dt": dt, "diag": np.array(diag), "stats": None, "vel": up, "vor": op, "pres": None,
                "delta": _s2p(e.dx(u[0]) + e.dy(u[1])), "spec": None, "num": None}
    diag, svor = e.run(q, case["steps"])
    return {"diag": diag, "svor": svor}
