"""Timing cases of the batched reactor-chemistry library on one GPU.

Every case calls the library as a program that uses it does: through the device-level handle
(zerork_hip.capi.Mech), the plugin API on host arrays (zerork_hip.capi.Plugin) or the learned
surrogate (zerork_hip.surrogate.Surrogate), on the seeded synthetic mechanisms that the tests
and the benchmark use (10, 53, 160 and 2,000 species).  Kinds of case:

  integrate   a batch of reactors advanced over one CFD time step, state resident on the GPU
  plugin      the same through zerork_reactor_solve, host arrays in and out, plugin defaults
  rates       dY/dt, dT/dt and the rates of progress of a batch of states
  jacobian    the analytic Jacobian of a batch of states
  forward     the surrogate's features and network on a batch of reactors (inference)
  gradients   the surrogate's forward and backward pass on one training batch

A case is a dict of plain values; listed() gives the named ones, draw(rng) one more of the same
ranges, prepare(case, seed) the inputs, run(state) one pass, work(case) its least traffic and
operations and exact(case, seed) the outputs from plain torch in 64 bits.
"""
import functools
import math
import os
import re
import sys

import numpy as np
import torch

ROOT = os.getcwd()
for _p in (ROOT, os.path.join(ROOT, "zero-rk_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from zerork_hip import capi, mechgen  # noqa: E402
from zerork_hip.surrogate import Surrogate  # noqa: E402

F64 = torch.float64


def listed():
    return [
        # one reactor state's derivatives: the least a caller can ask for (latency)
        dict(name="rates_10sp_1", kind="rates", mech="10sp", n=1),
        # the benchmark's rate-kernel batch: right-hand sides of an external integrator
        dict(name="rates_53sp_65536", kind="rates", mech="53sp", n=65536),
        # a detailed mechanism's right-hand sides
        dict(name="rates_2000sp_4096", kind="rates", mech="2000sp", n=4096),
        # Jacobians for an external implicit solver or a sensitivity analysis, ragged batch
        dict(name="jacobian_53sp_20001", kind="jacobian", mech="53sp", n=20001),
        # one CFD rank's cells through the plugin with its default solver options
        # (constant volume, SPGMR), host arrays in and out, a short CFD step
        dict(name="plugin_53sp_1500", kind="plugin", mech="53sp", n=1500, dt=1e-6),
        # the small-mechanism batch: fewer reactors than the GPU has room for, FP64
        dict(name="integrate_10sp_1024", kind="integrate", mech="10sp", n=1024, dt=1e-4,
             fp32=False, cvol=False),
        # the benchmark batch, the chosen method (FP32 Newton matrix)
        dict(name="integrate_53sp_65536", kind="integrate", mech="53sp", n=65536, dt=1e-4,
             fp32=True, cvol=False),
        # the plain FP64 method, constant volume, ragged batch, a shorter step
        dict(name="integrate_53sp_f64_9973", kind="integrate", mech="53sp", n=9973, dt=2e-5,
             fp32=False, cvol=True),
        # the medium mechanism (teams of wavefronts), FP32 Newton matrix
        dict(name="integrate_160sp_6000", kind="integrate", mech="160sp", n=6000, dt=1e-5,
             fp32=True, cvol=False),
        # the detailed mechanism (sparse Newton matrix)
        dict(name="integrate_2000sp_256", kind="integrate", mech="2000sp", n=256, dt=1e-6,
             fp32=True, cvol=False),
        # the surrogate's proposal for the benchmark's surrogate batch
        dict(name="forward_53sp_262144", kind="forward", mech="53sp", n=262144, hidden=256),
        # one step of the surrogate's training loop at its batch size
        dict(name="gradients_53sp_4096", kind="gradients", mech="53sp", n=4096, hidden=256),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_real(rng, lo, hi):
    return float("%.3g" % math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["rates", "rates", "jacobian", "plugin", "integrate", "integrate",
                       "integrate", "integrate", "forward", "gradients"])
    if kind == "rates":
        mech = rng.choice(["10sp", "53sp", "160sp", "2000sp"])
        top = {"10sp": 262144, "53sp": 65536, "160sp": 24576, "2000sp": 4096}[mech]
        return dict(kind=kind, mech=mech, n=_log_int(rng, 1, top))
    if kind == "jacobian":
        mech = rng.choice(["10sp", "53sp", "160sp"])
        top = {"10sp": 65536, "53sp": 32768, "160sp": 4096}[mech]
        return dict(kind=kind, mech=mech, n=_log_int(rng, 1, top))
    if kind == "plugin":
        return dict(kind=kind, mech=rng.choice(["10sp", "53sp"]), n=_log_int(rng, 1, 4096),
                    dt=_log_real(rng, 1e-7, 1e-5))
    if kind == "integrate":
        mech = rng.choice(["10sp", "53sp", "160sp", "2000sp"])
        if mech == "2000sp":
            return dict(kind=kind, mech=mech, n=_log_int(rng, 1, 256),
                        dt=_log_real(rng, 1e-8, 1e-6), fp32=True, cvol=rng.random() < 0.3)
        fp32 = rng.random() < 0.6
        top = {"10sp": 16384, "53sp": 32768, "160sp": 8192 if fp32 else 3000}[mech]
        return dict(kind=kind, mech=mech, n=_log_int(rng, 1, top),
                    dt=_log_real(rng, 1e-7, 1e-5 if mech == "160sp" else 1e-4), fp32=fp32,
                    cvol=rng.random() < 0.3)
    hidden = rng.choice([64, 128, 256])
    top = 262144 if kind == "forward" else 16384
    return dict(kind=kind, mech=rng.choice(["10sp", "53sp"]), n=_log_int(rng, 1, top),
                hidden=hidden)


# -- what a program holds ------------------------------------------------------------------
def _files(mech):
    d = os.path.join(ROOT, "tests", "golden", "mech", "synth_" + mech)
    return d + ".mech", d + ".therm"


@functools.lru_cache(None)
def _handle(mech):
    """The mechanism handle, loaded once by a program."""
    return capi.Mech(*_files(mech))


@functools.lru_cache(None)
def _generated(mech):
    return mechgen.workload_mechanism(mech)


@functools.lru_cache(None)
def _plugin(mech):
    p = capi.Plugin()
    for rc in (p.set_mechanism_files(*_files(mech)), p.set_double("rel_tol", 1e-6),
               p.set_double("abs_tol", 1e-12), p.load_mechanism()):
        if rc != 0:
            raise RuntimeError("plugin set-up failed (%d)" % rc)
    return p


def _states(case, seed):
    """The workload's initial states (fuel, oxidiser and products, no radicals)."""
    return mechgen.workload_states(case["mech"], _generated(case["mech"]), case["n"], seed)


def _dense(case, seed):
    """States in the middle of combustion: every species present."""
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    n, nsp = case["n"], _handle(case["mech"]).nsp
    u = lambda *s: torch.rand(*s, generator=g, device="cuda:0", dtype=F64)
    T = 800.0 + 1400.0 * u(n)
    P = 101325.0 * torch.exp(math.log(0.5) + math.log(80.0) * u(n))
    Y = -torch.log(u(n, nsp).clamp_min(1e-300))
    return T, P, Y / Y.sum(1, keepdim=True)


def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=F64, device="cuda:0")


def _surrogate(case, seed):
    """A network with the workload's normalisation, and n reactors with their own dt."""
    s = Surrogate(torch, _handle(case["mech"]), hidden=case["hidden"], seed=seed)
    g = torch.Generator(device="cpu").manual_seed(seed + 1)
    for b in s.net.b:
        b.copy_(0.1 * torch.randn(b.shape, generator=g))
    T, P, Y = _dense(case, seed)
    dt = torch.exp(torch.empty(case["n"], dtype=F64, device="cuda:0").uniform_(
        math.log(1e-6), math.log(1e-4),
        generator=torch.Generator(device="cuda:0").manual_seed(seed + 2)))
    x = _features64(T, P, Y, dt)
    s.mu[:s.nfeat] = x.mean(0).float()
    sd = x.std(0, unbiased=False).float()
    s.sig[:s.nfeat] = torch.where(sd > 1e-6, sd, torch.ones_like(sd))
    return s, T, P, Y, dt


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, n=case["n"])
    if kind in ("rates", "jacobian"):
        m = _handle(case["mech"])
        T, P, Y = _dense(case, seed)
        st.update(m=m, T=T, P=P, Y=Y)
        n, N = case["n"], m.nsp + 1
        new = lambda *s: torch.empty(*s, dtype=F64, device="cuda:0")
        if kind == "rates":
            st.update(ydot=new(n, N), rop=new(n, m.nstep))
        else:
            st.update(J=new(n, N, N), opts=capi.default_options())
    elif kind == "integrate":
        s = _states(case, seed)
        o = capi.default_options(rel_tol=1e-6, abs_tol=1e-12,
                                 fp32_preconditioner=int(case["fp32"]),
                                 constant_volume=int(case["cvol"]))
        if case["mech"] == "2000sp":  # the benchmark's step cap for this mechanism
            o.max_steps, o.cvode_num_retries = 1500, 1
        T, P, Y = _dev(s.T), _dev(s.P), _dev(s.Y)
        st.update(m=_handle(case["mech"]), opts=o, dt=case["dt"], T0=T, P0=P, Y0=Y,
                  T=T.clone(), P=P.clone(), Y=Y.clone())
    elif kind == "plugin":
        s = _states(case, seed)
        st.update(p=_plugin(case["mech"]), dt=case["dt"], T0=s.T, P0=s.P, Y0=s.Y)
    else:
        sur, T, P, Y, dt = _surrogate(case, seed)
        st.update(sur=sur)
        if kind == "forward":
            st.update(T=T, P=P, Y=Y, dt=dt)
        else:
            g = torch.Generator(device="cuda:0").manual_seed(seed + 3)
            target = torch.zeros(case["n"], sur.kout, device="cuda:0")
            target[:, :sur.nout] = torch.randn(case["n"], sur.nout, generator=g, device="cuda:0")
            st.update(X=sur.features(T, P, Y, dt), target=target)
    return st


def run(st):
    kind, n = st["kind"], st["n"]
    if kind == "rates":
        m = st["m"]
        m.rates(n, st["T"], st["P"], st["Y"], m.nsp, ydot=st["ydot"], rop=st["rop"])
        return {"ydot": st["ydot"], "rop": st["rop"]}
    if kind == "jacobian":
        m = st["m"]
        m.jacobian(n, st["T"], st["P"], st["Y"], m.nsp, st["J"], st["opts"])
        return {"J": st["J"]}
    if kind == "integrate":
        # the flow solver's new states of this step, then the chemistry
        m = st["m"]
        for k in ("T", "P", "Y"):
            st[k].copy_(st[k + "0"])
        m.integrate(n, st["dt"], st["T"], st["P"], st["Y"], m.nsp, st["opts"])
        return {"T": st["T"], "P": st["P"], "Y": st["Y"]}
    if kind == "plugin":
        T, P, Y = st["T0"].copy(), st["P0"].copy(), st["Y0"].copy()
        if st["p"].solve(0, 0.0, st["dt"], T, P, Y) != 0:
            raise RuntimeError("zerork_reactor_solve failed")
        return {"T": T, "P": P, "Y": Y}
    s = st["sur"]
    if kind == "forward":
        return {"out": s.forward(s.features(st["T"], st["P"], st["Y"], st["dt"]))}
    out, cache = s.forward(st["X"], cache=True)
    dout = torch.zeros_like(out)
    dout[:, :s.nout] = (out[:, :s.nout] - st["target"][:, :s.nout]) * (2.0 / (n * s.nout))
    dW, db = s.backward(dout, cache)
    return {"out": out, "dW": dW, "db": db}


# -- least traffic and operations ------------------------------------------------------------
_SIZES = {"10sp": (10, 27), "53sp": (53, 325), "160sp": (160, 900), "2000sp": (2000, 8000)}
# right-hand sides and Newton-matrix factorisations of a reactor of the workload over its dt
_RHS = {"10sp": (700, 60), "53sp": (260, 29), "160sp": (110, 20), "2000sp": (200, 25)}
_LU_FLOPS = {"2000sp": 2.0e6}


def work(case):
    n = case["n"]
    nsp, nrxn = _SIZES[case["mech"]]
    N, nstep = nsp + 1, 2 * nrxn
    rhs = 40.0 * nsp + 45.0 * nstep  # thermo; exponentials, products and sums of a step
    kind = case["kind"]
    if kind == "rates":
        return {"bytes": 8.0 * n * (nsp + 2 + N + nstep), "flops": n * rhs}
    if kind == "jacobian":
        return {"bytes": 8.0 * n * (nsp + 2 + N * N), "flops": n * (2 * rhs + 20.0 * nstep)}
    if kind in ("integrate", "plugin"):
        f, lu = _RHS[case["mech"]]
        one = f * (rhs + 2.0 * min(N * N, 90000)) + lu * _LU_FLOPS.get(case["mech"], 2.0 * N ** 3 / 3)
        return {"bytes": 16.0 * n * (nsp + 2), "flops": n * one}
    h = case["hidden"]
    kin, kout = (nsp + 18) // 16 * 16, (nsp + 16) // 16 * 16
    macs = kin * h + 2 * h * h + h * kout
    if kind == "forward":
        return {"bytes": n * (8.0 * (nsp + 3) + 4.0 * kout) + 2.0 * macs, "flops": 2.0 * n * macs}
    return {"bytes": n * (2.0 * kin + 8.0 * kout) + 6.0 * macs,
            "flops": n * (6.0 * macs - 2.0 * kin * h)}


# -- the outputs from plain torch in 64 bits ---------------------------------------------------
_RU, _PATM, _CAL = 8.314462618e3, 1.01325e5, 4184.0 / 8.314462618e3
_WT = {"H": 1.00794, "C": 12.0107, "N": 14.0067, "O": 15.9994, "AR": 39.948}


@functools.lru_cache(None)
def _tables(mech):
    """Numbers of a synthetic mechanism file: species weights and NASA-7 rows, Arrhenius
    parameters (kmol, m, K), participants, third-body and Troe data of its reactions."""
    mf, tf = _files(mech)
    body = re.sub(r"!.*", "", open(mf).read())
    species = re.search(r"SPECIES\s(.*?)\sEND", body, re.S).group(1).split()
    idx = {s: i for i, s in enumerate(species)}
    L = open(tf).read().splitlines()
    mw, nasa = np.zeros(len(species)), np.zeros((len(species), 14))
    for k, l in enumerate(L):
        if len(l) >= 80 and l[79] == "1" and l.split()[0] in idx:
            i = idx[l.split()[0]]
            for c in range(24, 44, 5):
                e = l[c:c + 2].strip()
                if e:
                    mw[i] += _WT[e] * int(l[c + 2:c + 5])
            t = "".join(x[:75] for x in L[k + 1:k + 4])
            nasa[i] = [float(t[15 * q:15 * q + 15]) for q in range(14)]
    rx = []
    for l in body[body.index("REACTIONS"):].splitlines()[1:]:
        if "<=>" in l:
            f = l.rsplit(None, 3)
            tb, fo = "+ M" in f[0], "(+M)" in f[0]
            sides = [[idx[s] for s in re.sub(r"\(\+M\)|\+ M\b", "", q).replace("+", " ").split()]
                     for q in f[0].split("<=>")]
            rx.append(dict(r=sides[0], p=sides[1], k=[float(v) for v in f[1:]], tb=tb, fo=fo,
                           low=None, troe=None, eff={}))
        elif l.strip().startswith("LOW"):
            rx[-1]["low"] = [float(v) for v in l.split("/")[1].split()]
        elif l.strip().startswith("TROE"):
            rx[-1]["troe"] = [float(v) for v in l.split("/")[1].split()]
        elif "/" in l:
            rx[-1]["eff"] = {idx[a]: float(b) for a, b in re.findall(r"(\S+?)/\s*([^/\s]+)\s*/", l)}
    return species, mw, nasa, rx


class _Chem:
    """Rates of a batch of states at constant pressure in 64 bits."""

    def __init__(self, mech):
        self.dev = "cuda:0" if torch.cuda.is_available() else "cpu"
        sp, mw, nasa, rx = _tables(mech)
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=F64, device=self.dev)
        self.nsp, self.mw, self.nasa, self.nr = len(sp), t(mw), t(nasa), len(rx)
        A = [(math.log(r["k"][0] * 1e-3 ** (len(r["r"]) - 1 + r["tb"])), r["k"][1],
              r["k"][2] * _CAL) for r in rx]
        self.arr = t(A).T
        pad = lambda v: v + [len(sp)] * (4 - len(v))
        self.re = torch.as_tensor([pad(r["r"]) for r in rx], device=self.dev)
        self.pr = torch.as_tensor([pad(r["p"]) for r in rx], device=self.dev)
        self.dn = t([len(r["p"]) - len(r["r"]) for r in rx])
        self.is_tb = torch.as_tensor([r["tb"] for r in rx], device=self.dev)
        self.fo = [j for j, r in enumerate(rx) if r["fo"]]
        self.enh = [j for j, r in enumerate(rx) if r["fo"] or r["tb"]]
        eff = np.zeros((len(self.enh), len(sp)))
        for q, j in enumerate(self.enh):
            for s, v in rx[j]["eff"].items():
                eff[q, s] = v - 1.0
        self.eff = t(eff)
        low = [(math.log(rx[j]["low"][0] * 1e-3 ** len(rx[j]["r"])), rx[j]["low"][1],
                rx[j]["low"][2] * _CAL) for j in self.fo]
        self.low = t(low).T if low else None
        # three-parameter Troe has no fourth term: exp(-inf) = 0
        self.troe = t([(rx[j]["troe"] + [math.inf])[:4] for j in self.fo]).T if low else None
        self.steps = {}

    def thermo(self, T):
        a = torch.where((T < 1000.0)[:, None, None], self.nasa[None, :, 7:], self.nasa[None, :, :7])
        T = T[:, None]
        cp = a[..., 0] + T * (a[..., 1] + T * (a[..., 2] + T * (a[..., 3] + T * a[..., 4])))
        h = (a[..., 0] + T * (a[..., 1] / 2 + T * (a[..., 2] / 3 + T * (a[..., 3] / 4 +
             T * a[..., 4] / 5))) + a[..., 5] / T)
        s = (a[..., 0] * torch.log(T) + T * (a[..., 1] + T * (a[..., 2] / 2 + T * (a[..., 3] / 3 +
             T * a[..., 4] / 4))) + a[..., 6])
        return cp, h, h - s

    def k_of(self, p, T):
        return torch.exp(p[0] + p[1] * torch.log(T)[:, None] - p[2] / T[:, None])

    def rhs(self, T, P, Y):
        """ydot [n, nsp + 1], rop [n, 2 reactions] (forward, reverse), cp, h/RT, density and
        the concentrations."""
        n = len(T)
        cp, h, g = self.thermo(T)
        rho = P / (_RU * T * (Y / self.mw).sum(1))
        C = rho[:, None] * Y / self.mw
        one = torch.ones(n, 1, dtype=F64, device=self.dev)
        C1, G0 = torch.cat([C, one], 1), torch.cat([g, 0 * one], 1)
        kf = self.k_of(self.arr, T)
        dG = G0[:, self.re].sum(2) - G0[:, self.pr].sum(2)
        kr = kf * torch.exp(-(self.dn * torch.log(_PATM / (_RU * T))[:, None]) - dG)
        if self.enh:
            M = C.sum(1, keepdim=True) + C @ self.eff.T
            full = torch.ones_like(kf)
            full[:, self.enh] = M
            mul = torch.where(self.is_tb, full, torch.ones_like(full))
            if self.fo:
                Pr = (self.k_of(self.low, T) * full[:, self.fo] / kf[:, self.fo]).clamp_min(1e-300)
                a, t3, t1, t2 = self.troe
                t = T[:, None]
                Fc = ((1 - a) * torch.exp(-t / t3) + a * torch.exp(-t / t1) +
                      torch.exp(-t2 / t)).clamp_min(1e-300)
                f, lp = torch.log10(Fc), torch.log10(Pr)
                x = lp - (0.4 + 0.67 * f)
                x = x / (0.75 - 1.27 * f - 0.14 * x)
                mul[:, self.fo] = 10.0 ** (f / (1 + x * x)) * Pr / (1 + Pr)
            kf, kr = kf * mul, kr * mul
        lim = 1.0e22
        kf, kr = kf * (lim / (lim + kf)), kr * (lim / (lim + kr))
        rf, rr = kf * C1[:, self.re].prod(2), kr * C1[:, self.pr].prod(2)
        q = rf - rr
        net = torch.zeros(n, self.nsp + 1, dtype=F64, device=self.dev)
        for k in range(4):
            net.index_add_(1, self.pr[:, k], q)
            net.index_add_(1, self.re[:, k], -q)
        net = net[:, :self.nsp]
        cpm = cp * _RU / self.mw
        cpx = (cpm * Y).sum(1)
        Td = -(h * net).sum(1) / rho * _RU * T / cpx
        ydot = torch.cat([net * self.mw / rho[:, None], Td[:, None]], 1)
        return ydot, torch.stack([rf, rr], 2).reshape(n, -1), cpm, cpx, h, rho, C

    def jacobian(self, T, P, Y):
        """The reference's approximate Jacobian: concentration derivatives of the rates of
        progress at frozen third bodies and density, the temperature row from the species block,
        the temperature column a forward difference."""
        n, ns = len(T), self.nsp
        f0, rop, cpm, cpx, h, rho, C = self.rhs(T, P, Y)
        dT = (T + T * 2.0 ** -26) - T
        f1 = self.rhs(T + dT, P, Y)[0]
        J = torch.zeros(n, ns + 1, ns + 1, dtype=F64, device=self.dev)
        flat = J.view(n, -1)
        inv = torch.cat([1.0 / C, torch.zeros(n, 1, dtype=F64, device=self.dev)], 1)
        for d, (a, b) in enumerate(((self.re, self.pr), (self.pr, self.re))):
            for k in range(4):
                v = rop[:, d::2] * inv[:, a[:, k]]
                for q in range(4):  # absent participants (index ns) land in the row and column
                    flat.index_add_(1, a[:, q] * (ns + 1) + a[:, k], -v)  # overwritten below
                    flat.index_add_(1, b[:, q] * (ns + 1) + a[:, k], v)
        S = J[:, :ns, :ns]
        row = (S * h[:, :, None]).sum(1) * (_RU * T)[:, None] + f0[:, ns:] * cpm * self.mw
        J[:, ns, :ns] = -row / self.mw / cpx[:, None]
        S *= self.mw[None, :, None] / self.mw[None, None, :]
        J[:, :, ns] = (f1 - f0) / dT[:, None]
        return J


@functools.lru_cache(None)
def _chem(mech):
    return _Chem(mech)


def _features64(T, P, Y, dt):
    return torch.cat([torch.log(T)[:, None], torch.log(P)[:, None],
                      torch.log(Y.clamp_min(1e-20)), torch.log(dt)[:, None]], 1)


def _gelu64(z):
    return 0.5 * z * (1 + torch.erf(z * math.sqrt(0.5)))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("integrate", "plugin"):
        return None  # a converged integration of the batch takes minutes
    st = prepare(case, seed)
    if kind in ("rates", "jacobian"):
        c = _chem(case["mech"])
        T, P, Y = st["T"], st["P"], st["Y"]
        some = max(1, int(2e8) // (2 * c.nr + c.nsp * 14 + (c.nsp + 1) ** 2))
        got = []
        for i in range(0, case["n"], some):
            s = slice(i, i + some)
            r = c.rhs(T[s], P[s], Y[s])[:2] if kind == "rates" else (c.jacobian(T[s], P[s], Y[s]),)
            got.append(r)
        out = [torch.cat(v) for v in zip(*got)]
        return dict(zip(("ydot", "rop") if kind == "rates" else ("J",), out))
    s = st["sur"]
    W = [w.double() for w in s.net.W]
    B = [b.double() for b in s.net.b]
    if kind == "forward":
        x = torch.zeros(case["n"], s.kin, dtype=F64, device="cuda:0")
        x[:, :s.nfeat] = _features64(st["T"], st["P"], st["Y"], st["dt"])
        h = (x - s.mu.double()) / s.sig.double()
        h[:, s.nfeat:] = 0.0
    else:
        h = st["X"].double()
    hs, zs = [h], []
    for i, (w, b) in enumerate(zip(W, B)):
        z = h @ w + b
        h = z if i == len(W) - 1 else _gelu64(z)
        zs.append(z)
        hs.append(h)
    if kind == "forward":
        return {"out": h}
    d = torch.zeros_like(h)
    d[:, :s.nout] = (h - st["target"].double())[:, :s.nout] * (2.0 / (case["n"] * s.nout))
    dW, db = [None] * len(W), [None] * len(W)
    for i in range(len(W) - 1, -1, -1):
        dW[i], db[i] = hs[i].T @ d, d.sum(0)
        if i:
            z = zs[i - 1]
            d = (d @ W[i].T) * (0.5 * (1 + torch.erf(z * math.sqrt(0.5))) +
                                z * torch.exp(-0.5 * z * z) / math.sqrt(2 * math.pi))
    return {"out": hs[-1], "dW": dW, "db": db}
