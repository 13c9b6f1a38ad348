"""Performance cases of the time-domain LISA response: the calls a user's program makes, over the
range of sizes and options they are made at, with the same numbers in plain 64-bit torch.

A case is a dict of plain values:
    path       "dropin"   pyResponseTDI.get_projections + get_tdi_delays on a resident series
               "wrapper"  ResponseWrapper(GBWave()) called with source parameters
               "batch"    BatchedResponse plan of many sources of uneven length, plan.run()
               "inner"    one sampler step: BatchPlan.rebind to new sky positions, then the fused
                          inner products with a data series and the log-likelihoods
    n          samples of the source (batch and inner: of the longest allowed source)
    sources    number of sources (batch and inner)
    dt         sampling interval (s)
    orbits     "equal" (equal-arm cartwheel) or "cartwheel" (six unequal, time-varying arms)
    tdi        "1st generation", "2nd generation" or "sagnac" (a combination given as a list)
    chan       "AET" or "XYZ"
    order      Lagrange interpolation order
    precision  "fp64", "mixed" (complex64 input), "mixed-q31" or "mixed-c128"
    exact      the reference's stencil operation order (fp64) or the division-free stencils
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lisa-on-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

YRSID_SI = 31558149.763545603
C_SI = 299792458.0
C_INV = 3.3356409519815204e-09
AU_SI = 149597870700.0
ARM = 2.5e9
T_BUFFER = 10000.0
ORBIT_SPAN = 2.0 * YRSID_SI
ORBIT_DT = 1.0e4
YEAR = 3_153_600  # samples of a year at dt = 10 s
LINKS = (12, 23, 31, 13, 32, 21)

# The Sagnac combination alpha (light sent around the constellation both ways), as the list of
# terms of channel X that pyResponseTDI takes; Y and Z follow cyclically.
SAGNAC = [
    {"link": 12, "links_for_delay": [], "sign": 1},
    {"link": 23, "links_for_delay": [12], "sign": 1},
    {"link": 31, "links_for_delay": [12, 23], "sign": 1},
    {"link": 13, "links_for_delay": [], "sign": -1},
    {"link": 32, "links_for_delay": [13], "sign": -1},
    {"link": 21, "links_for_delay": [13, 32], "sign": -1},
]


def _case(name, path, n, sources=1, dt=10.0, orbits="equal", tdi="2nd generation", chan="AET",
          order=25, precision="fp64", exact=True):
    c = {"path": path, "n": int(n), "sources": int(sources), "dt": dt, "orbits": orbits,
         "tdi": tdi, "chan": chan, "order": order, "precision": precision,
         "exact": bool(exact) and precision == "fp64"}
    return dict(name=name, **c) if name else c


def listed():
    return [
        # a merger's last day, as a sampler calls it for every proposal: the call itself counts
        _case("short_wrapper", "wrapper", 8192),
        # the CPU configuration of the reference's own documentation: 1st generation
        _case("dropin_2e17_1st", "dropin", 131072, tdi="1st generation"),
        # the year-long galactic binary, FP64 drop-in as the reference runs it (the default)
        _case("dropin_year", "dropin", YEAR),
        # the same on arms that differ and change, which any realistic orbit file gives
        _case("dropin_year_unequal", "dropin", YEAR, orbits="cartwheel"),
        # a third of a year, the division-free FP64 stencils (exact=False), an odd length
        _case("dropin_fast", "dropin", 1_000_003, exact=False),
        # year-long source from its parameters to A, E, T with float32 outputs
        _case("wrapper_year_c128", "wrapper", YEAR, precision="mixed-c128"),
        # the 8-byte input format: packed from the caller's complex128 series on every call
        _case("dropin_mixed", "dropin", 1 << 20, precision="mixed"),
        # a user's own combination with another interpolation order: the general kernels
        _case("sagnac_order31", "dropin", 262_145, orbits="cartwheel", tdi="sagnac", chan="XYZ",
              order=31),
        # a catalogue: 64 binaries of uneven duration, one fused launch
        _case("batch_c128", "batch", YEAR, sources=64, precision="mixed-c128"),
        # a smaller catalogue on unequal arms
        _case("batch_c128_unequal", "batch", 1 << 20, sources=8, orbits="cartwheel",
              precision="mixed-c128"),
        # a catalogue in FP64, bitwise the drop-in
        _case("batch_fp64", "batch", 500_000, sources=16),
        # one step of 32 walkers: new sky positions, inner products with the data, likelihoods
        _case("inner_walkers", "inner", 1 << 17, sources=32, precision="mixed-c128"),
    ]


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, n | 1 if rng.random() < 0.6 else n))


def draw(rng):
    path = rng.choice(["dropin", "dropin", "dropin", "wrapper", "batch", "batch", "inner"])
    dt = rng.choice([5.0, 10.0])
    orbits = rng.choice(["equal", "equal", "cartwheel"])
    tdi = rng.choice(["1st generation", "2nd generation", "2nd generation"])
    chan = rng.choice(["AET", "AET", "XYZ"])
    lo = 8192 if dt == 10.0 else 12000
    if path == "inner":
        return _case(None, path, _log_int(rng, 32768, 1 << 18), sources=rng.randint(4, 48), dt=dt,
                     orbits=orbits, tdi=tdi,
                     precision=rng.choice(["mixed", "mixed-c128", "mixed-c128"]))
    precision = rng.choice(["fp64", "fp64", "mixed-c128", "mixed", "mixed-q31"])
    exact = rng.random() < 0.7
    if path == "batch":
        precision = rng.choice(["fp64", "mixed-c128", "mixed-c128"])
        return _case(None, path, _log_int(rng, 1 << 16, 1 << 20), sources=rng.randint(3, 32),
                     dt=dt, orbits=orbits, tdi=tdi, chan=chan, precision=precision, exact=exact)
    n = _log_int(rng, lo, YEAR)
    order = 25
    if path == "dropin" and precision == "fp64" and rng.random() < 0.3:
        order = rng.choice([15, 31])
        tdi = rng.choice([tdi, "sagnac"])
    if path == "wrapper":
        n = _gb_length(n, dt)
    return _case(None, path, n, dt=dt, orbits=orbits, tdi=tdi, chan=chan, order=order,
                 precision=precision, exact=exact)


# ------------------------------------------------------------------ inputs

def _lengths(case):
    """Uneven durations, U[0.05, 1] of the longest (inner: all alike, as a sampler's walkers)."""
    if case["path"] == "inner":
        return [case["n"]] * case["sources"]
    r = random.Random(case["n"] * 1009 + case["sources"])
    least = int(2 * T_BUFFER / case["dt"]) + 1500
    return [max(least, int(r.uniform(0.05, 1.0) * case["n"])) for _ in range(case["sources"])]


def _gb_length(n, dt):
    """A number of samples from n on that the wrapper's observation time reproduces."""
    while len(np.arange(0.0, (n * (1 / (1 / dt))) / YRSID_SI * YRSID_SI, dt)) != n:
        n += 1
    return n


def _sources(case, seed):
    """Galactic binaries of mHz frequencies: (A, f0, fdot, iota, phi0, psi) and (lam, beta)."""
    rng = np.random.default_rng([int(seed), 20])
    m = case["sources"]
    par = np.stack([10 ** rng.uniform(-22, -21, m), 10 ** rng.uniform(-2.7, -2.1, m),
                    10 ** rng.uniform(-18, -16, m), np.arccos(rng.uniform(-0.9, 0.9, m)),
                    rng.uniform(0, 2 * np.pi, m), rng.uniform(0, 2 * np.pi, m)], axis=1)
    lam = rng.uniform(0, 2 * np.pi, m)
    beta = np.arcsin(rng.uniform(-0.95, 0.95, m))
    return par, lam, beta


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _waveform(p, n, dt):
    """h+ + i hx of one galactic binary (complex128)."""
    A, f, fdot, iota, phi0, psi = (float(x) for x in p)
    t = torch.arange(n, dtype=torch.float64, device=_device()) * dt
    fddot = 11.0 / 3.0 * fdot ** 2 / f
    tt = t * t
    phase = 2 * math.pi * ((f * t + 0.5 * fdot * tt) + (1.0 / 6.0) * fddot * (tt * t)) - phi0
    ci = math.cos(iota)
    hs = -torch.cos(phase) * A * (1.0 + ci * ci)
    hc = -torch.sin(phase) * 2.0 * A * ci
    c2, s2 = math.cos(2 * psi), math.sin(2 * psi)
    return torch.complex(hs * c2 - hc * s2, hs * s2 + hc * c2)


def _data(case, seed, total):
    """The data series of a sampler: noise of the signals' size, float32, laid out as outputs."""
    g = torch.Generator(device=_device()).manual_seed(int(seed) * 7 + 3)
    return torch.randn(3 * total, generator=g, device=_device(), dtype=torch.float32) * 1e-21


_ORBITS = {}


def _orbits(kind):
    from fastlisaresponse_amd.orbits import CartwheelOrbits, EqualArmlengthOrbits
    if kind not in _ORBITS:
        cls = EqualArmlengthOrbits if kind == "equal" else CartwheelOrbits
        o = cls(armlength=ARM, t_max=ORBIT_SPAN, dt_base=ORBIT_DT)
        o.configure(linear_interp_setup=True)
        _ORBITS[kind] = o
    return _ORBITS[kind]


def prepare(case, seed):
    par, lam, beta = _sources(case, seed)
    orbits = _orbits(case["orbits"])
    tdi = SAGNAC if case["tdi"] == "sagnac" else case["tdi"]
    fs, n = 1 / case["dt"], case["n"]
    kw = dict(order=case["order"], tdi=tdi, orbits=orbits, tdi_chan=case["chan"],
              exact=case["exact"], precision=case["precision"])
    st = {"path": case["path"], "case": case}
    if case["path"] == "dropin":
        from fastlisaresponse_amd import pyResponseTDI
        st["model"] = pyResponseTDI(fs, n, **kw)
        st["h"] = _waveform(par[0], n, case["dt"])
        st["sky"] = (float(lam[0]), float(beta[0]))
    elif case["path"] == "wrapper":
        from fastlisaresponse_amd import ResponseWrapper
        from fastlisaresponse_amd.waveforms import GBWave
        st["wrap"] = ResponseWrapper(GBWave(), n * case["dt"] / YRSID_SI, case["dt"], 6, 7,
                                     t_buffer=T_BUFFER, remove_sky_coords=True, n_overide=n, **kw)
        st["args"] = [float(x) for x in par[0]] + [float(lam[0]), float(beta[0])]
    else:
        from fastlisaresponse_amd.batch import BatchedResponse, pack_mixed, pack_q31
        lengths = _lengths(case)
        h = torch.cat([_waveform(p, m, case["dt"]) for p, m in zip(par, lengths)])
        scales = None
        if case["precision"] == "mixed":
            h, scales = pack_mixed(h, lengths)
        elif case["precision"] == "mixed-q31":
            h, scales = pack_q31(h, lengths)
        br = BatchedResponse(fs, t_buffer=T_BUFFER, **kw)
        st["plan"] = br.plan(h, lengths, lam, beta, scales=scales)
        st["sky"], st["scales"], st["lengths"] = (lam, beta), scales, lengths
        if case["path"] == "inner":
            from fastlisaresponse_amd.utility import data_sums
            st["data"] = _data(case, seed, sum(lengths))
            st["dsums"] = data_sums(st["data"], lengths, st["plan"].offsets, br.tdi_start_ind)
    return st


def run(st):
    if st["path"] == "dropin":
        m = st["model"]
        m.get_projections(st["h"], *st["sky"], t0=0.0, t_buffer=T_BUFFER)
        out = list(m.get_tdi_delays())
        return {"tdi": out, "y": m.y_gw} if st["case"]["precision"] == "fp64" else {"tdi": out}
    if st["path"] == "wrapper":
        return list(st["wrap"](*st["args"]))
    plan = st["plan"]
    if st["path"] == "batch":
        plan.run()
        return plan.out_all
    from fastlisaresponse_amd.utility import log_likelihood_from_sums
    plan.rebind(*st["sky"], scales=st["scales"])
    sums = plan.inner_products(st["data"])
    return {"sums": sums, "loglike": log_likelihood_from_sums(sums, st["dsums"], 1e-42)}


# ------------------------------------------------------------------ work

def work(case):
    """Each input read once, each output written once; a complex stencil per receiving and per
    emitting spacecraft (per link where the arms differ) and a real one per TDI term, two
    operations per tap."""
    total = sum(_lengths(case)) if case["path"] in ("batch", "inner") else case["n"]
    mixed = case["precision"] != "fp64"
    hb = 8 if case["precision"] in ("mixed", "mixed-q31") and case["path"] != "dropin" else 16
    if case["path"] == "wrapper":
        hb = 0
    ob = 3 * (4 if mixed else 8)
    if case["path"] == "dropin" and not mixed:
        ob += 6 * 8
    taps = case["order"] + 1
    units = {"1st generation": 24, "2nd generation": 48, "sagnac": 18}[case["tdi"]]
    stencils = 6 if case["orbits"] == "equal" else 9
    return {"bytes": total * (hb + ob), "flops": total * taps * (4 * stencils + 2 * units)}


# ------------------------------------------------------------------ the same in 64 bits

def _tables(kind):
    """Orbit tables of the cartwheel constellation on t = k * ORBIT_DT: positions [N, 3, 3] and
    light travel times [N, 6]."""
    def pos(t):
        a = 2.0 * np.pi * t / YRSID_SI + 0.0
        ecc = ARM / (2.0 * np.sqrt(3.0) * AU_SI)
        x = np.zeros((len(t), 3, 3))
        for i in range(3):
            b = 2.0 * np.pi * i / 3.0 + 0.0
            x[:, i, 0] = AU_SI * np.cos(a) + 0.5 * ecc * AU_SI * (np.cos(2 * a - b) - 3 * np.cos(b))
            x[:, i, 1] = AU_SI * np.sin(a) + 0.5 * ecc * AU_SI * (np.sin(2 * a - b) - 3 * np.sin(b))
            x[:, i, 2] = -np.sqrt(3.0) * ecc * AU_SI * np.cos(a - b)
        return x
    base = np.arange(0.0, ORBIT_SPAN + 0.5 * ORBIT_DT, ORBIT_DT)
    t = np.arange(0.0, base.max() + 0.5 * ORBIT_DT, ORBIT_DT)
    t = t[t <= base.max()]
    x = pos(t)
    ltt = np.full((len(t), 6), ARM / C_SI)
    if kind != "equal":
        for r, link in enumerate(LINKS):
            i, j = divmod(link, 10)
            L = np.linalg.norm(x[:, i - 1] - x[:, j - 1], axis=-1) / C_SI
            for _ in range(3):
                L = np.linalg.norm(x[:, i - 1] - pos(t - L)[:, j - 1], axis=-1) / C_SI
            ltt[:, r] = L
    return x, ltt


class _Exact:
    """Projections and TDI of one configuration in 64-bit torch: linear interpolation in the orbit
    tables, Lagrange stencils with the tabulated prefactor A(e), sums in the combination's order."""

    def __init__(self, case):
        self.case, self.dev = case, _device()
        self.fs = 1 / case["dt"]
        self.dt = 1 / self.fs
        x, ltt = _tables(case["orbits"])
        self.rmax = float(np.sqrt(np.sum(x * x, axis=-1)).max())
        cols = np.concatenate([ltt, x.reshape(len(x), 9)], axis=1)
        self.val = torch.as_tensor(cols.T.copy(), device=self.dev)
        self.slope = torch.as_tensor(((cols[1:] - cols[:-1]) / ORBIT_DT).T.copy(), device=self.dev)
        h = self.h = (case["order"] + 1) // 2
        fact = [float(math.factorial(k)) for k in range(2 * h + 2)]
        self.deps = 1.0 / 1000
        eps = np.arange(1001) * self.deps
        A = np.ones(1001)
        for i in range(1, h):
            A = A * ((i + eps) * (i + 1 - eps))
        self.A = torch.as_tensor(A / (fact[h - 1] * fact[h]), device=self.dev)
        self.E = [(fact[h - 1] / fact[h - 1 - j]) * (fact[h] / fact[h + j]) * (-1.0) ** j
                  for j in range(1, h)]
        self.T = int(T_BUFFER / self.dt)
        self.P = self.T - 2 * (int(100.0 * self.fs) + 4 * case["order"])

    def node(self, t):
        k = torch.clamp((t / ORBIT_DT).to(torch.int64), 0, self.val.shape[1] - 2)
        return k, t - ORBIT_DT * k.to(torch.float64)

    def col(self, node, c):
        k, tau = node
        return self.slope[c][k] * tau + self.val[c][k]

    def split(self, delay, t0):
        cf = (delay - t0) * self.fs
        d = torch.ceil(cf).to(torch.int64) - 1
        return d, (1.0 + d.to(torch.float64)) - cf

    def stencil(self, rows, d, e):
        """The stencil at sample d, fraction e of each row."""
        ind = torch.clamp((e / self.deps).to(torch.int64), 0, 999)
        f = (e - ind.to(torch.float64) * self.deps) / self.deps
        A = self.A[ind] * (1.0 - f) + self.A[ind + 1] * f
        D = e * (1.0 - e)
        sums = [torch.zeros_like(e) for _ in rows]
        for j in range(1, self.h):
            F, G = j + e, j + (1 - e)
            for s, x in zip(sums, rows):
                s += self.E[j - 1] * (x[d + 1 + j] / F + x[d - j] / G)
        return [A * ((1.0 - e) * x[d + 1] + e * x[d] + D * s) for s, x in zip(sums, rows)]

    @staticmethod
    def dot(a, b):
        return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2]

    def projections(self, h, lam, beta, t0=0.0):
        n, dev = h.shape[0], self.dev
        cb, sb, cl, sl = np.cos(beta), np.sin(beta), np.cos(lam), np.sin(lam)
        k, u, v = (-cb * cl, -cb * sl, -sb), (sl, -cl, 0.0), (-sb * cl, -sb * sl, cb)
        rows = [h.real.contiguous(), h.imag.contiguous()]
        y = torch.zeros((6, n), dtype=torch.float64, device=dev)
        i = torch.arange(self.P, n - self.P, dtype=torch.float64, device=dev)
        t = t0 + i * self.dt
        nr = self.node(t)
        rec = {}
        for s in range(3):
            x = [self.col(nr, 6 + 3 * s + c) for c in range(3)]
            rec[s] = (x, self.stencil(rows, *self.split(t - self.dot(k, x) * C_INV, t0)))
        shared = {}
        for r, link in enumerate(LINKS):
            s, e = link // 10 - 1, link % 10 - 1
            key = e if self.case["orbits"] == "equal" else link
            if key not in shared:
                te = t - self.col(nr, r)
                ne = self.node(te)
                xe = [self.col(ne, 6 + 3 * e + c) for c in range(3)]
                shared[key] = (xe, self.stencil(rows, *self.split(te - self.dot(k, xe) * C_INV, t0)))
            (xr, hr), (xe, he) = rec[s], shared[key]
            nv = [a - b for a, b in zip(xr, xe)]
            norm = torch.sqrt(self.dot(nv, nv))
            nv = [a / norm for a in nv]
            un, vn = self.dot(u, nv), self.dot(v, nv)
            xp, xc = 0.5 * (un * un - vn * vn), un * vn
            y[r, self.P:n - self.P] = (1.0 / (1.0 - self.dot(k, nv))) * (
                (he[0] - hr[0]) * xp + (he[1] - hr[1]) * xc)
        return y

    def terms(self):
        if self.case["tdi"] == "sagnac":
            return [(t["link"], tuple(t["links_for_delay"]), t["sign"]) for t in SAGNAC]
        first = [(13, (), 1), (31, (13,), 1), (12, (13, 31), 1), (21, (13, 31, 12), 1),
                 (12, (), -1), (21, (12,), -1), (13, (12, 21), -1), (31, (12, 21, 13), -1)]
        second = [(12, (13, 31, 12, 21), 1), (21, (13, 31, 12, 21, 12), 1),
                  (13, (13, 31, 12, 21, 12, 21), 1), (31, (13, 31, 12, 21, 12, 21, 13), 1),
                  (13, (12, 21, 13, 31), -1), (31, (12, 21, 13, 31, 13), -1),
                  (12, (12, 21, 13, 31, 13, 31), -1), (21, (12, 21, 13, 31, 13, 31, 12), -1)]
        return first if self.case["tdi"] == "1st generation" else first + second

    def tdi(self, y, t0=0.0):
        n = y.shape[1]
        out = torch.zeros((3, n), dtype=torch.float64, device=self.dev)
        i = torch.arange(self.T, n - self.T, dtype=torch.float64, device=self.dev)
        t = t0 + i * self.dt
        nd = self.node(t)
        L = {link: self.col(nd, r) for r, link in enumerate(LINKS)}
        for c in range(3):
            def cyc(link):
                return 10 * ((link // 10 - 1 + c) % 3 + 1) + (link % 10 - 1 + c) % 3 + 1
            acc = torch.zeros_like(t)
            for link, chain, sign in self.terms():
                delay = t
                for q in chain:
                    delay = delay - L[cyc(q)]
                acc += sign * self.stencil([y[LINKS.index(cyc(link))]], *self.split(delay, t0))[0]
            out[c, self.T:n - self.T] = acc
        if self.case["chan"] == "XYZ":
            return out
        X, Y, Z = out
        return torch.stack([(Z - X) / math.sqrt(2.0), (X - 2.0 * Y + Z) / math.sqrt(6.0),
                            (X + Y + Z) / math.sqrt(3.0)])


def exact(case, seed):
    par, lam, beta = _sources(case, seed)
    ex = _Exact(case)
    lengths = _lengths(case) if case["path"] in ("batch", "inner") else [case["n"]]
    outs, y = [], None
    for s, n in enumerate(lengths):
        y = ex.projections(_waveform(par[s], n, case["dt"]), lam[s], beta[s])
        outs.append(ex.tdi(y))
    if case["path"] == "dropin":
        out = {"tdi": list(outs[0])}
        return dict(out, y=y) if case["precision"] == "fp64" else out
    if case["path"] == "wrapper":
        return [c[ex.T:-ex.T] for c in outs[0]]
    if case["path"] == "batch":
        return torch.cat([o.reshape(-1) for o in outs])
    total = sum(lengths)
    data = _data(case, seed, total).double()
    sums, loglike, at = [], [], 0
    for o, n in zip(outs, lengths):
        d = data[3 * at:3 * (at + n)].view(3, n)[:, ex.T:n - ex.T]
        v = o[:, ex.T:n - ex.T]
        alt = torch.ones(v.shape[1], dtype=torch.float64, device=v.device)
        alt[1::2] = -1.0
        sums.append(torch.stack([(d * v).sum(1), (v * v).sum(1), v.sum(1), (v * alt).sum(1)], dim=1))
        loglike.append(-0.5 * ((d - v).square().sum(1) / 1e-42).sum())
        at += n
    return {"sums": torch.stack(sums), "loglike": torch.stack(loglike)}
