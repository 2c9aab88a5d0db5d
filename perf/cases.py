"""The calls a user of this library times: what a lattice-QCD program has the GPU do on one gauge field.

A program generates (or reads) a configuration, keeps it resident, and then
solves M x = b on it for point sources (propagators) or noise sources
(disconnected loops), in the precision and with the solver it chose.  Every
case goes through the package's public calls with the host arrays they take.
Extents are multiples of 4, as the library asks.

kind        call                                       stands for
hop         diracops.Hsingle                           one hopping term of a host program's own algorithm
schur       diracops.Hdbletm                           the even-odd operator, Wilson or twisted mass
bicgstab    quark.fermprop(inverter=0)                 a point-source solve without deflation
gmresdr     quark.fermprop(inverter=5)                 a point-source solve by GMRES-DR in FP64
psc         quark.fermprop(inverter=6) twice           a noise source by GMRES-DR, the next over its deflation space
mixed       inverters.solve_mixed                      the even-odd solve with FP32 or FP16 inner precision
propagator  quark.propagator                           the spin-colour sources of one site, solved together
noise       disconloops.noise_loop                     the disconnected-loop estimate from Z4 sources
smear       diracops.smear                             Gaussian smearing of a source or sink
heatbath    diracops.gauge_heatbath                    gauge-field generation, and the field back on the host

The gauge field of a case is its configuration: thermalised once by the
library's heatbath and kept resident, as a program keeps it, while sources
change from call to call.  ``heatbath`` generates a new one in every pass.
"""
import math

import numpy as np
import torch

from baylorlqcd_amd import diracops, disconloops, inverters, lattice, quark

BETA = 6.0
THERMALISE = 200  # sweeps from a random field to the configuration of a case
BC = (1, 1, 1, -1)


# ---- the cases ------------------------------------------------------------

def listed():
    return [
        # one hopping term on the smallest lattice in use: launches, copies and call overhead
        dict(name="hop_8x8x8x16", kind="hop", nx=8, ny=8, nz=8, nt=16, idag=0, parity=2),
        # the twisted-mass operator on a production-size field held by the host
        dict(name="schur_24x24x24x48", kind="schur", nx=24, ny=24, nz=24, nt=48, kappa=0.156, mu=0.005, idag=1),
        # the small-lattice solves of the reference's own first configuration
        dict(name="bicgstab_8x8x8x16", kind="bicgstab", nx=8, ny=8, nz=8, nt=16, kappa=0.150, mu=0.0),
        dict(name="gmresdr_12x8x20x28", kind="gmresdr", nx=12, ny=8, nz=20, nt=28, kappa=0.150, mu=0.0, m=40, k=10),
        # the FP64 solver where the basis no longer fits any cache
        dict(name="gmresdr_24x24x24x48", kind="gmresdr", nx=24, ny=24, nz=24, nt=48, kappa=0.1535, mu=0.0, m=40,
             k=16),
        # first and second right-hand side of a deflated sequence, twisted mass
        dict(name="psc_16x16x16x32", kind="psc", nx=16, ny=16, nz=16, nt=32, kappa=0.154, mu=0.005, m=60, k=20),
        # the mixed-precision solver: FP32 on an ordinary lattice, FP16 on the largest
        dict(name="mixed32_16x16x16x32", kind="mixed", nx=16, ny=16, nz=16, nt=32, kappa=0.1545, mu=0.0, m=40, k=16,
             basis=1, prec=1, recon=18),
        dict(name="mixed16_32x32x32x64", kind="mixed", nx=32, ny=32, nz=32, nt=64, kappa=0.1565, mu=0.0, m=40, k=16,
             basis=2, prec=2, recon=12),
        # many right-hand sides: a whole point propagator, and a noise estimate
        dict(name="propagator_12x20x16x24", kind="propagator", nx=12, ny=20, nz=16, nt=24, kappa=0.154, mu=0.003,
             m=40, k=16, nrhs=12),
        dict(name="noise_16x16x16x32", kind="noise", nx=16, ny=16, nz=16, nt=32, kappa=0.1545, mu=0.0, m=60, k=20,
             nrhs=24),
        # both ends of a run: source smearing, gauge generation
        dict(name="smear_16x16x16x32", kind="smear", nx=16, ny=16, nz=16, nt=32, nsmear=40, asmear=0.08),
        dict(name="heatbath_24x24x24x48", kind="heatbath", nx=24, ny=24, nz=24, nt=48, nsweep=10),
    ]


#: Largest number of sites that draw() gives a kind: no drawn case costs more than the largest listed one.
MOST_SITES = {"hop": 2 << 20, "schur": 2 << 20, "bicgstab": 1 << 18, "gmresdr": 1 << 19, "psc": 1 << 18,
              "mixed": 1 << 20, "propagator": 1 << 17, "noise": 1 << 17, "smear": 1 << 20, "heatbath": 1 << 20}


def draw(rng):
    kind = rng.choice(sorted(MOST_SITES))
    least, most = 4096, MOST_SITES[kind]
    want = math.exp(rng.uniform(math.log(least), math.log(most)))
    while True:
        side = want ** 0.25
        n = [4 * max(1, round(side * math.exp(rng.uniform(-0.5, 0.5)) / 4)) for _ in range(3)]
        n.append(4 * max(1, round(want / (n[0] * n[1] * n[2]) / 4)))
        v = n[0] * n[1] * n[2] * n[3]
        if least // 2 <= v <= most and max(n) <= 96:
            break
    c = dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], nt=n[3])
    if kind == "hop":
        c.update(idag=rng.randint(0, 1), parity=rng.randint(1, 2))
    elif kind == "smear":
        c.update(nsmear=rng.randint(1, 60), asmear=round(rng.uniform(0.03, 0.12), 3))
    elif kind == "heatbath":
        c.update(nsweep=rng.randint(1, 12))
    else:
        # a small volume's lowest modes fluctuate: it is used at heavier quarks
        c.update(kappa=round(rng.uniform(0.146, 0.152 if v < 1 << 15 else 0.1545), 4),
                 mu=rng.choice([0.0, round(rng.uniform(0.001, 0.02), 4)]))
        if kind == "schur":
            c.update(idag=rng.randint(0, 1))
        elif kind != "bicgstab":
            m, k = rng.choice([(20, 5), (30, 8), (40, 10), (40, 16), (50, 15), (60, 20)])
            c.update(m=m, k=k)
    if kind == "mixed":
        basis, prec = rng.choice([(1, 1), (1, 2), (2, 2)])
        c.update(basis=basis, prec=prec, recon=rng.choice([12, 18]))
    elif kind == "propagator":
        c.update(nrhs=rng.choice([3, 12]))
    elif kind == "noise":
        c.update(nrhs=rng.randint(2, 24))
    return c


# ---- inputs ---------------------------------------------------------------

def _dims(c):
    return c["nx"], c["ny"], c["nz"], c["nt"]


def _coact():
    co = np.zeros((4, 4, 4), order="F")
    co[2, :2, :] = 1.0
    return co


def _spinor_len(n):
    nvh = n[0] * n[1] * n[2] * n[3] // 32
    return 6 * (nvh + max(2 * nvh // m for m in n)) * 64


_field = {"n": None, "u": None}  # the configuration this program keeps resident


def _configuration(n):
    """The links of the case's lattice, resident; the host array identifies them in later calls."""
    if _field["n"] != n or _field["u"] is None:
        _field.update(n=None, u=None)
        lattice.init(n, BC)
        diracops.gauge_heatbath(BETA, THERMALISE, 2024, 1, _coact())
        u = diracops.gauge_get_ref(n)
        diracops.gauge_load(u, _coact())
        _field.update(n=n, u=u)
    return _field["u"]


def _random_spinor(n, gen, z4=False):
    """A reference-layout checkerboard of Gaussian or Z4 noise (the rows past nvhalf carry no data)."""
    nvh = n[0] * n[1] * n[2] * n[3] // 32
    a = torch.zeros(8, 2, 4, _spinor_len(n) // 384, 3, 2, dtype=torch.float64, device="cuda")
    if z4:
        r = torch.randint(0, 4, (8, 2, 4, nvh, 3), generator=gen, device="cuda")
        a[:, :, :, :nvh, :, 0] = (r == 0).double() - (r == 1).double()
        a[:, :, :, :nvh, :, 1] = (r == 2).double() - (r == 3).double()
    else:
        a[:, :, :, :nvh] = torch.randn(8, 2, 4, nvh, 3, 2, generator=gen, device="cuda", dtype=torch.float64)
    return a.reshape(-1).cpu().numpy()


def prepare(case, seed):
    n, kind = _dims(case), case["kind"]
    s = dict(case=case, n=n, seed=seed, coact=_coact(), bc=BC)
    if kind == "heatbath":
        if _field["n"] != n or _field["u"] is not None:
            lattice.init(n, BC)
            _field.update(n=n, u=None)
        return s
    s["u"] = _configuration(n)
    if "kappa" in case:
        s["kappa"] = (case["kappa"], case["mu"])
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    pick = np.random.default_rng(seed)
    empty = lambda: np.zeros(_spinor_len(n))  # noqa: E731
    if kind in ("hop", "schur", "mixed"):
        s["b"], s["x"] = _random_spinor(n, gen), empty()
    elif kind == "smear":
        s["b"] = [_random_spinor(n, gen) for _ in range(2)]
        s["x"] = [empty(), empty()]
    elif kind in ("bicgstab", "gmresdr"):
        s["b"], s["x"] = [empty(), empty()], [empty(), empty()]
        site = [int(pick.integers(1, m + 1)) for m in n]
        quark.pointsource(s["b"][0], s["b"][1], site, int(pick.integers(1, 4)), int(pick.integers(1, 5)))
    elif kind == "psc":
        s["b"] = [_random_spinor(n, gen, z4=True) for _ in range(4)]
        s["x"] = [empty() for _ in range(4)]
    elif kind == "propagator":
        s["site"] = tuple(int(pick.integers(1, m + 1)) for m in n)
    return s


def _fermprop(s, inverter, i, isignal=1):
    c = s["case"]
    m, k = (c["m"], c["k"]) if inverter else (1, 0)  # BiCGStab: 1 = from the constant vector
    be, bo, xe, xo = s["b"][2 * i], s["b"][2 * i + 1], s["x"][2 * i], s["x"][2 * i + 1]
    quark.fermprop("", be, bo, -1, s["kappa"], 0.0, inverter, s["coact"], s["bc"], 1e-10, 0, 1.0, s["u"], m, k, xe,
                   xo, isignal=isignal)


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "hop":
        diracops.Hsingle(s["x"], s["u"], s["b"], c["idag"], s["coact"], s["bc"], c["parity"])
    elif kind == "schur":
        diracops.Hdbletm(s["x"], s["u"], None, s["b"], c["idag"], s["coact"], s["kappa"], -1, s["bc"])
    elif kind == "bicgstab":
        _fermprop(s, 0, 0)
    elif kind == "gmresdr":
        _fermprop(s, 5, 0)
    elif kind == "psc":
        _fermprop(s, 6, 0, isignal=1)
        _fermprop(s, 6, 1, isignal=2)
    elif kind == "mixed":
        s["x"].fill(0.0)
        inverters.solve_mixed(s["b"], s["x"], (c["m"], c["k"]), 1e-10, c["basis"], c["prec"], c["recon"], 0.0, 0,
                              s["u"], s["coact"], s["kappa"], s["bc"])
    elif kind == "propagator":
        p = quark.propagator(c["nrhs"], s["site"], s["kappa"], (c["m"], c["k"]), 1e-10, solutions=True)
        return p["xe"] + p["xo"]
    elif kind == "noise":
        r = disconloops.noise_loop(c["nrhs"], s["seed"], s["kappa"], (c["m"], c["k"]), 1e-10, coact=s["coact"],
                                   bc=s["bc"], u=s["u"])
        return [r["traces"], r["loops"]]
    elif kind == "smear":
        diracops.smear(s["x"][0], s["x"][1], s["u"], s["b"][0], s["b"][1], c["asmear"], c["nsmear"], s["bc"])
    elif kind == "heatbath":
        diracops.gauge_heatbath(BETA, c["nsweep"], s["seed"], 0, s["coact"])
        return diracops.gauge_get_canonical(s["n"])
    return s["x"]


# ---- what a pass cannot do without, and how exact it is --------------------

def _steps(c):
    """Krylov steps that a solve at this hopping parameter takes, roughly (beta = 6.0, 1e-10)."""
    return 2.0 / (1.0 / c["kappa"] - 1.0 / 0.1575) ** 0.9 + 60


def work(case):
    """Bytes: the links and the host arrays, once each.  Flops: the operator applications of the solves."""
    v = _dims(case)[0] * _dims(case)[1] * _dims(case)[2] * _dims(case)[3]
    links, half, hop = v * 576, v * 96, v // 2 * 1320
    kind = case["kind"]
    if kind in ("hop", "schur"):
        return dict(bytes=links + 2 * half, flops=hop * (1 if kind == "hop" else 2))
    if kind == "smear":
        return dict(bytes=links * 3 // 4 + 4 * half, flops=case["nsmear"] * v * 6 * 4 * 72)
    if kind == "heatbath":
        return dict(bytes=2 * links, flops=case["nsweep"] * v * 4 * (6 * 2 * 198 + 1500))
    nrhs = {"psc": 2}.get(kind, case.get("nrhs", 1))
    fields = {"mixed": 2, "noise": 0, "propagator": 2}.get(kind, 4)
    return dict(bytes=links + nrhs * fields * half, flops=nrhs * _steps(case) * 2 * hop)


def tolerance(case):
    """Operators: FP64 sums in another order.  Solves stop on a residual, so solutions agree to that residual
    times the system's condition: 1e-10 of the start, which for BiCGStab is the constant vector and not the point
    source; psc's second solve stops at 1e-8, as the reference's."""
    tight, solve = {"rel": 2e-15, "max": 5e-14}, {"rel": 1e-7, "max": 1e-5}
    return {"hop": tight, "schur": tight, "smear": tight, "heatbath": {"rel": 1e-12, "max": 1e-10},
            "bicgstab": {"rel": 2e-6, "max": 2e-4}, "psc": {"rel": 1e-6, "max": 1e-4},
            "noise": {"rel": 2e-10, "max": 2e-8}}.get(case["kind"], solve)


# ---- the same in torch, in 64 bits ------------------------------------------

def _gammas():
    g = torch.zeros(4, 4, 4, dtype=torch.complex128, device="cuda")
    for r in range(4):
        g[0, r, 3 - r] = 1
        g[1, r, 3 - r] = (-1j, 1j, -1j, 1j)[r]
        g[2, r, (r + 2) % 4] = (1, -1, 1, -1)[r]
        g[3, r, r] = (1, 1, -1, -1)[r]
    return g


def _slots(n):
    """Canonical site of every reference slot, [parity][block pair, parity in block, row]."""
    nvh = n[0] * n[1] * n[2] * n[3] // 32
    ns = [m // 2 for m in n]
    out = []
    for par in range(2):
        block = [b for b in range(16) if bin(b).count("1") % 2 == par]
        site = torch.zeros(8, 2, nvh, dtype=torch.int64)
        for q, b in enumerate(block):
            for e in range(2):
                w = 2 * torch.arange(nvh)
                x = [w % ns[0], w // ns[0] % ns[1], w // (ns[0] * ns[1]) % ns[2], w // (ns[0] * ns[1] * ns[2])]
                x[0] = x[0] + ((x[0] + x[1] + x[2] + x[3]) % 2 != e)
                g = [2 * x[m] + ((b >> m) & 1) for m in range(4)]
                site[q, e] = g[0] + n[0] * (g[1] + n[1] * (g[2] + n[2] * g[3]))
        out.append(site.cuda())
    return out


class _Exact:
    """The operators on whole fields [t, z, y, x, spin, colour]."""

    def __init__(self, n, u=None):
        self.n, self.v = n, n[0] * n[1] * n[2] * n[3]
        self.grid = (n[3], n[2], n[1], n[0])
        self.g = _gammas()
        self.g5 = self.g[0] @ self.g[1] @ self.g[2] @ self.g[3]
        self.slots = _slots(n)
        if u is not None:
            nvh = self.v // 32
            w = torch.from_numpy(u).reshape(16, 2, 4, -1, 9, 2)[:, :, :, :nvh].cuda()
            self.u = torch.zeros(self.v, 4, 9, dtype=torch.complex128, device="cuda")
            for par in range(2):
                block = [b for b in range(16) if bin(b).count("1") % 2 == par]
                self.u[self.slots[par]] = torch.view_as_complex(w[block].permute(0, 1, 3, 2, 4, 5).contiguous())
            self.u = self.u.reshape(*self.grid, 4, 3, 3)

    def parity(self, par):
        p = sum(torch.arange(m, device="cuda").reshape([-1 if i == k else 1 for i in range(4)])
                for k, m in enumerate(self.grid)) % 2 == par
        return p[..., None, None]

    def field(self, even=None, odd=None):
        f = torch.zeros(self.v, 4, 3, dtype=torch.complex128, device="cuda")
        for a, s in ((even, self.slots[0]), (odd, self.slots[1])):
            if a is not None:
                w = torch.from_numpy(a).reshape(8, 2, 4, -1, 3, 2)[:, :, :, :self.v // 32].cuda()
                f[s] = torch.view_as_complex(w.permute(0, 1, 3, 2, 4, 5).contiguous())
        return f.reshape(*self.grid, 4, 3)

    def host(self, f, par):
        a = torch.zeros(8, 2, 4, _spinor_len(self.n) // 384, 3, 2, dtype=torch.float64, device="cuda")
        a[:, :, :, :self.v // 32] = torch.view_as_real(f.reshape(self.v, 4, 3)[self.slots[par]]).permute(0, 1, 3, 2, 4, 5)
        return a.reshape(-1).cpu().numpy()

    def times(self, u, f):
        """u f over colour at every site."""
        return sum(u[..., None, :, c] * f[..., :, None, c] for c in range(3))

    def shift(self, f, mu, forward):
        """f(x + mu) or f(x - mu), times the boundary condition on the hop across the edge."""
        f = torch.roll(f, -1 if forward else 1, 3 - mu)
        if BC[mu] != 1:
            f.select(3 - mu, self.n[mu] - 1 if forward else 0).mul_(BC[mu])
        return f

    def transport(self, f, mu, forward):
        u = self.u.select(-3, mu)
        return self.times(u, self.shift(f, mu, True)) if forward else \
            self.shift(self.times(u.mH, f), mu, False)

    def spin(self, g, f):
        return torch.einsum("ab,tzyxbc->tzyxac", g, f)

    def hop(self, f, dagger=0):
        one, out = torch.eye(4, dtype=torch.complex128, device="cuda"), torch.zeros_like(f)
        sign = -1 if dagger else 1
        for mu in range(4):
            out += self.spin(one - sign * self.g[mu], self.transport(f, mu, True))
            out += self.spin(one + sign * self.g[mu], self.transport(f, mu, False))
        return out

    def schur(self, f, kappa, mu, dagger=0):
        a = 2 * kappa * mu
        tw = 1j * self.g5
        t = self.hop(f, dagger) * self.parity(1)
        t = self.hop(t - a * self.spin(tw, t), dagger) * self.parity(0)
        return (f + a * self.spin(tw, f)) / kappa ** 2 - t / (1 + a * a)

    def solve(self, b, op):
        """BiCGStab to rounding, restarted from the true residual."""
        x, dot = torch.zeros_like(b), lambda p, q: torch.vdot(p.reshape(-1), q.reshape(-1))
        bn = float(b.norm())
        for _ in range(4):
            r = b - op(x)
            if float(r.norm()) < 2e-14 * bn:
                break
            rh, p, v, rho, alpha, omega = r.clone(), 0 * r, 0 * r, 1.0, 1.0, 1.0
            goal = max(float(r.norm()) * 1e-12, 1e-14 * bn)
            for it in range(4000):
                rho, old = dot(rh, r), rho
                p = r + rho / old * alpha / omega * (p - omega * v)
                v = op(p)
                alpha = rho / dot(rh, v)
                r = r - alpha * v
                t = op(r)
                omega = dot(t, r) / dot(t, t)
                x += alpha * p + omega * r
                r = r - omega * t
                if it % 8 == 7 and float(r.norm()) < goal:
                    break
        return x

    def full(self, kappa, mu):
        tw = 2j * kappa * mu * self.g5
        return lambda f: f + self.spin(tw, f) - kappa * self.hop(f)


def _mix(z):
    """The splitmix64 finaliser on int64 tensors."""
    shift = lambda a, k: (a >> k) & ((1 << (64 - k)) - 1)  # noqa: E731
    z = (z ^ shift(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ shift(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ shift(z, 31)


GOLDEN = 0x9E3779B97F4A7C15 - (1 << 64)


def _z4(e, seed, r):
    """Noise source r of the noise loop."""
    c = torch.arange(e.v * 12, device="cuda") + r * e.v * 12
    u = ((_mix(seed + GOLDEN * (1 + c)) >> 11) & ((1 << 53) - 1)).double() / 2.0 ** 53
    re = (u > 0.75).double() - ((u > 0.5) & (u < 0.75)).double()
    im = ((u > 0.25) & (u < 0.5)).double() - ((u <= 0.25) | (u == 0.5) | (u == 0.75)).double()
    return torch.complex(re, im).reshape(*e.grid, 4, 3)


def _loops(e, kappa, eta, x):
    """Traces of the 16 local matrices and the nine loop operators, per timeslice."""
    one, g, g5 = torch.eye(4, dtype=torch.complex128, device="cuda"), e.g, e.g5
    mats = [one, *g, g5, *(a @ g5 for a in g)]
    mats += [0.5j * (g[a] @ g[b] - g[b] @ g[a]) for a in range(4) for b in range(a + 1, 4)]
    per_t = lambda a, b: (a.conj() * b).sum((1, 2, 3, 4, 5))  # noqa: E731
    traces = torch.stack([per_t(eta, e.spin(m, x)) for m in mats], 1)
    ops = []
    for mu in range(4):
        u = e.u.select(-3, mu)
        back = per_t(e.shift(x, mu, True), e.spin(one - g[mu], e.times(u.mH, eta)))
        ops.append(kappa * (back - per_t(x, e.spin(one + g[mu], e.transport(eta, mu, True)))).conj())
    ops += [per_t(x, eta).conj()] + [per_t(x, e.spin(g[mu], eta)).conj() for mu in range(4)]
    loops = torch.zeros(e.n[3], 5, 9, dtype=torch.complex128, device="cuda")
    loops[:, 0] = torch.stack(ops, 1)
    return traces, loops


def _heatbath(n, nsweep, seed):
    """Cabibbo-Marinari / Kennedy-Pendleton sweeps from the unit field, draws from the counter-based stream."""
    v, vh = n[0] * n[1] * n[2] * n[3], n[0] * n[1] * n[2] * n[3] // 2
    u = torch.eye(3, dtype=torch.complex128, device="cuda").expand(v, 4, 3, 3).contiguous()
    golden = lambda z: _mix(z + GOLDEN)  # noqa: E731
    q = 2 * torch.arange(vh, device="cuda")
    x = [q % n[0], q // n[0] % n[1], q // (n[0] * n[1]) % n[2], q // (n[0] * n[1] * n[2])]

    def site(y):
        y = [y[m] % n[m] for m in range(4)]
        return y[0] + n[0] * (y[1] + n[1] * (y[2] + n[2] * y[3]))

    def mul(a, b):
        return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)

    for sweep in range(nsweep):
        for par in range(2):
            xs = [x[0] + (par + x[1] + x[2] + x[3]) % 2, *x[1:]]
            here = site(xs)
            for mu in range(4):
                to = lambda **d: site([xs[m] + d.get("f", {}).get(m, 0) for m in range(4)])  # noqa: E731
                staple = 0
                for nu in range(4):
                    if nu == mu:
                        continue
                    up = mul(mul(u[to(f={mu: 1}), nu], u[to(f={nu: 1}), mu].mH), u[here, nu].mH)
                    down, far = to(f={nu: -1}), to(f={mu: 1, nu: -1})
                    staple = staple + up + mul(u[far, nu].mH, mul(u[down, mu].mH, u[down, nu]))
                w = u[here, mu]
                state = golden(torch.arange(vh, device="cuda") + ((sweep * 8 + par * 4 + mu) << 32))
                state = golden(state ^ seed)

                def uniform(use):
                    nonlocal state
                    state = torch.where(use, golden(state), state)
                    return (((state >> 11) & ((1 << 53) - 1)).double() + 1.0) / 2.0 ** 53

                for p, r in ((0, 1), (1, 2), (0, 2)):
                    m = mul(w, staple)
                    a = [0.5 * (m[:, p, p].real + m[:, r, r].real), 0.5 * (m[:, p, r].imag + m[:, r, p].imag),
                         0.5 * (m[:, p, r].real - m[:, r, p].real), 0.5 * (m[:, p, p].imag - m[:, r, r].imag)]
                    k = sum(t * t for t in a).sqrt()
                    alpha, x0 = 2.0 * BETA * k / 3.0, torch.ones_like(k)
                    todo = torch.ones_like(k, dtype=torch.bool)
                    for _ in range(200):
                        r1, r2, r3, r4 = (uniform(todo) for _ in range(4))
                        big = -(r1.log() + torch.cos(6.283185307179586 * r2) ** 2 * r3.log()) / alpha
                        good = todo & (r4 * r4 <= 1.0 - 0.5 * big)
                        x0 = torch.where(good, 1.0 - big, x0)
                        todo = todo & ~good
                        if not bool(todo.any()):
                            break
                    every = torch.ones_like(todo)
                    rad = (1.0 - x0 * x0).clamp(min=0).sqrt()
                    ct = 2.0 * uniform(every) - 1.0
                    ph = 6.283185307179586 * uniform(every)
                    st = (1.0 - ct * ct).clamp(min=0).sqrt()
                    y = [x0, rad * st * ph.cos(), rad * st * ph.sin(), rad * ct]
                    b = [t / k for t in a]
                    c0 = sum(s * t for s, t in zip(y, b))
                    c1 = -y[0] * b[1] + b[0] * y[1] + (y[2] * b[3] - y[3] * b[2])
                    c2 = -y[0] * b[2] + b[0] * y[2] + (y[3] * b[1] - y[1] * b[3])
                    c3 = -y[0] * b[3] + b[0] * y[3] + (y[1] * b[2] - y[2] * b[1])
                    wp, wr = w[:, p].clone(), w[:, r].clone()
                    w[:, p] = torch.complex(c0, c3)[:, None] * wp + torch.complex(c2, c1)[:, None] * wr
                    w[:, r] = torch.complex(-c2, c1)[:, None] * wp + torch.complex(c0, -c3)[:, None] * wr
                w[:, 0] /= w[:, 0].norm(dim=1, keepdim=True)
                w[:, 1] -= (w[:, 0].conj() * w[:, 1]).sum(1, keepdim=True) * w[:, 0]
                w[:, 1] /= w[:, 1].norm(dim=1, keepdim=True)
                w[:, 2] = torch.linalg.cross(w[:, 0], w[:, 1]).conj()
                u[here, mu] = w
    return u.cpu().numpy()


def exact(case, seed):
    n, kind = _dims(case), case["kind"]
    v = n[0] * n[1] * n[2] * n[3]
    if kind == "heatbath":
        return _heatbath(n, case["nsweep"], seed)
    if "m" in case and v * case.get("nrhs", 1) > 4 << 20 or kind == "mixed" and v > 1 << 20:
        return None  # minutes of solves
    s = prepare(case, seed)
    e = _Exact(n, s["u"])
    if kind == "hop":
        f = e.field(odd=s["b"]) if case["parity"] == 1 else e.field(even=s["b"])
        return e.host(e.hop(f, case["idag"]), case["parity"] - 1)
    if kind == "smear":
        f = e.field(*s["b"])
        for _ in range(case["nsmear"]):
            f = (1 - 6 * case["asmear"]) * f + case["asmear"] * sum(
                e.transport(f, mu, d) for mu in range(3) for d in (True, False))
        return [e.host(f, 0), e.host(f, 1)]
    kappa, mu = s["kappa"]
    mu = 0.0 if kind in ("schur", "mixed") and mu < 1e-8 else mu
    if kind == "schur":
        return e.host(e.schur(e.field(even=s["b"]), kappa, mu, case["idag"]), 0)
    if kind == "mixed":
        return e.host(e.solve(e.field(even=s["b"]), lambda f: e.schur(f, kappa, mu)), 0)
    op = e.full(kappa, mu)
    if kind == "noise":
        total = [0, 0]
        for r in range(case["nrhs"]):
            eta = _z4(e, seed, r)
            total = [a + b / case["nrhs"] for a, b in zip(total, _loops(e, kappa, eta, e.solve(eta, op)))]
        return [a.cpu().numpy() for a in total]
    if kind == "propagator":
        out = []
        for r in range(case["nrhs"]):
            b = torch.zeros(*e.grid, 4, 3, dtype=torch.complex128, device="cuda")
            px, py, pz, pt = (m - 1 for m in s["site"])
            b[pt, pz, py, px, r // 3, r % 3] = 1
            out.append(e.solve(b, op))
        return [e.host(f, 0) for f in out] + [e.host(f, 1) for f in out]
    out = []
    for i in range(len(s["b"]) // 2):
        f = e.solve(e.field(s["b"][2 * i], s["b"][2 * i + 1]), op)
        out += [e.host(f, 0), e.host(f, 1)]
    return out
