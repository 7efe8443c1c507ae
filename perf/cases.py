"""The work that users of this framework have it do, as cases to be timed.

listed() names the cases, draw(rng) makes more of the same ranges, prepare()
makes what a program holds before the call, run() makes one pass through the
public entry points of mattohf_amd.tdhf, work() counts what a pass cannot do
without, and exact() evaluates the same outputs with plain torch in FP64
(complex128), from the definitions: the pair transforms of the Fock exchange
one by one, the gradients by torch's own differentiation.

Cells: acell grows with NG as in the repository's tests and benchmark, with a
time step that RK4 holds stable there.
"""
import math

import numpy as np
import torch

from mattohf_amd import tdhf as T

# acell, ion charge and RK4 time step per grid size (the reference's example
# cell at NG=16, the tests' and the benchmark's cells otherwise)
CELLS = {16: (3.6, 1.0, 0.02), 32: (8.0, 4.0, 0.025), 64: (10.0, 8.0, 0.01),
         128: (12.0, 16.0, 0.004)}


def listed():
    return [
        # one H|w> of a small cell, called from a host program: latency
        {"name": "hpsi_ng32_nk4", "kind": "hpsi", "ng": 32, "nk": 4, "nb": 2, "nbocc": 2},
        # one RK4 step per call (a program with its own time loop), odd sizes
        {"name": "step_ng64_nk21", "kind": "step", "ng": 64, "nk": 21, "nb": 3, "nbocc": 3},
        # linear response of the reference's example system: empty bands, kick
        {"name": "rt_ng16_nk40", "kind": "rt", "ng": 16, "nk": 40, "nb": 8, "nbocc": 1,
         "nt": 200, "field": "kick"},
        # laser runs of the small, the ordinary and the largest cell
        {"name": "rt_ng32_nk32", "kind": "rt", "ng": 32, "nk": 32, "nb": 2, "nbocc": 2,
         "nt": 200, "field": "pulse"},
        {"name": "rt_ng64_nk64", "kind": "rt", "ng": 64, "nk": 64, "nb": 4, "nbocc": 4,
         "nt": 100, "field": "pulse"},
        {"name": "rt_ng128_nk128", "kind": "rt", "ng": 128, "nk": 128, "nb": 8, "nbocc": 8,
         "nt": 8, "field": "pulse"},
        # a few small trajectories together, ragged k-meshes, no tuning
        {"name": "batch_ng32_small", "kind": "batch", "ng": 32, "nks": "7,12,20", "ntraj": 6,
         "nb": 2, "nbocc": 2, "nt": 50, "tune": False},
        # a pulse scan over three k-meshes, tuned once as the benchmark does
        {"name": "batch_ng64_mixed", "kind": "batch", "ng": 64, "nks": "16,32,64", "ntraj": 48,
         "nb": 4, "nbocc": 4, "nt": 50, "tune": True},
        # gradient of the final energy with respect to the field (pulse shaping)
        {"name": "grad_ng32_nk32", "kind": "grad", "ng": 32, "nk": 32, "nb": 2, "ntraj": 1,
         "nt": 200, "objective": "energy"},
        # gradients of the emitted current for several pulses of the largest cell
        {"name": "grad_ng128_nk128", "kind": "grad", "ng": 128, "nk": 128, "nb": 8, "ntraj": 3,
         "nt": 4, "objective": "jsq"},
        # the first iterations of a ground state (Krylov, Rayleigh-Ritz)
        {"name": "gs_ng64_nk64", "kind": "gs", "ng": 64, "nk": 64, "nb": 4, "nbocc": 4,
         "ncg": 4, "nscf": 5},
        # spectra after a run
        {"name": "spectrum_20000", "kind": "spectrum", "nt": 20000, "nomega": 4000, "window": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hpsi", "step", "rt", "rt", "batch", "batch", "grad", "grad", "gs",
                       "spectrum"])
    ng = rng.choice([16, 32, 64, 128])
    nk = _log_int(rng, 3, 128)
    nb = rng.randint(1, 8)
    nbocc = nb if rng.random() < 0.6 else rng.randint(1, nb)
    if kind in ("hpsi", "step"):
        return {"kind": kind, "ng": ng, "nk": nk, "nb": nb, "nbocc": nbocc}
    if kind == "rt":
        return {"kind": kind, "ng": ng, "nk": nk, "nb": nb, "nbocc": nbocc,
                "nt": min(_log_int(rng, 8, 250), _steps_for(ng, nk, nb, nbocc, 6e11)),
                "field": rng.choice(["pulse", "kick"])}
    if kind == "batch":
        ng = rng.choice([16, 32, 64])
        nks = [_log_int(rng, 4, 64) for _ in range(rng.randint(1, 3))]
        nb, ntraj = rng.randint(1, 4), _log_int(rng, 2, 48)
        return {"kind": kind, "ng": ng, "nks": ",".join(map(str, nks)), "ntraj": ntraj, "nb": nb,
                "nbocc": nb, "nt": _log_int(rng, 10, 60), "tune": rng.random() < 0.5}
    if kind == "grad":
        nk, nb, ntraj = _log_int(rng, 3, 96), rng.randint(1, 6), rng.randint(1, 4)
        cap = _steps_for(ng, nk, nb, nb, 1e11) // ntraj
        return {"kind": kind, "ng": ng, "nk": nk, "nb": nb, "ntraj": ntraj,
                "nt": max(2, min(_log_int(rng, 4, 200), cap)),
                "objective": rng.choice(["energy", "jsq"])}
    if kind == "gs":
        ng = rng.choice([16, 32, 64])
        nb, ncg = rng.randint(1, 5), rng.randint(2, 4)
        while nb * ncg > min(16, ng // 2):
            nb -= 1
        return {"kind": kind, "ng": ng, "nk": _log_int(rng, 4, 64), "nb": nb,
                "nbocc": rng.randint(1, nb), "ncg": ncg, "nscf": rng.randint(2, 5)}
    return {"kind": kind, "nt": _log_int(rng, 500, 20000), "nomega": _log_int(rng, 100, 4000),
            "window": rng.randint(0, 1)}


# ---------------------------------------------------------------------------
# work of a pass
# ---------------------------------------------------------------------------
def _h_flops(ng, nk, nb, nbocc):
    """FP64 operations of one H application by the pair transforms of the
    reference algorithm (5 N log2 N per transform)."""
    f = 5.0 * ng * math.log2(ng)
    pairs = nk * nk * nb * nbocc
    return pairs * (16 * ng + 2 * f) + nb * nk * (2 * f + 20 * ng) + 2 * f + nk * nbocc * 4 * ng


def _steps_for(ng, nk, nb, nbocc, flops):
    return max(2, int(flops / (4 * _h_flops(ng, nk, nb, nbocc))))


def _nks(case):
    given = [int(k) for k in case["nks"].split(",")]
    return [given[t % len(given)] for t in range(case["ntraj"])]


def work(case):
    k = case["kind"]
    if k == "spectrum":
        return {"bytes": 8 * (4 * case["nt"] + 7 * case["nomega"]),
                "flops": case["nt"] * case["nomega"] * 30}
    ng, nb = case["ng"], case["nb"]
    nbocc = case.get("nbocc", nb)
    if k == "batch":
        h = sum(_h_flops(ng, n, nb, nbocc) for n in _nks(case))
        state = 16 * ng * nb * sum(_nks(case))
        return {"bytes": 2 * state + 5 * 8 * case["ntraj"] * case["nt"],
                "flops": 4 * case["nt"] * h}
    h, state = _h_flops(ng, case["nk"], nb, nbocc), 16 * ng * nb * case["nk"]
    if k == "hpsi":
        return {"bytes": 3 * state, "flops": h}
    if k == "step":
        return {"bytes": 2 * state, "flops": 4 * h}
    if k == "rt":
        return {"bytes": 2 * state + 5 * 8 * case["nt"], "flops": 4 * case["nt"] * h}
    if k == "grad":  # a reverse stage costs two forward ones
        return {"bytes": case["ntraj"] * (3 * state + 5 * 8 * case["nt"]),
                "flops": 12 * case["ntraj"] * case["nt"] * h}
    return {"bytes": 2 * state, "flops": case["nscf"] * (2 * case["ncg"] + 1) * h}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _orbitals(rs, ng, nb, nk, acell):
    """Smooth orthonormal orbitals (NG, NB, NK): plane waves with amplitudes
    that fall off as those of a ground state do."""
    g = np.fft.fftfreq(ng, 1.0 / ng)
    fall = np.exp(-0.5 * np.abs(g) * min(1.0, 16.0 / ng))
    c = fall * (rs.standard_normal((nk, nb, ng)) + 1j * rs.standard_normal((nk, nb, ng)))
    u = np.fft.ifft(c, axis=2)
    q, _ = np.linalg.qr(u.transpose(0, 2, 1))
    return np.asfortranarray(q.transpose(1, 2, 0) / math.sqrt(acell / ng))


def _field(rs, nt, dt, kind):
    """A and Aave of nt steps: the impulsive kick, or a window of a sin^2
    pulse well inside its envelope."""
    if kind == "kick":
        _, A, Aave, _ = T.define_afield_lr(nt, dt, float(rs.uniform(0.5e-4, 2e-4)))
        return A, Aave
    A0 = math.exp(rs.uniform(math.log(0.01), math.log(0.5)))
    om, cep = rs.uniform(0.03, 0.10), rs.uniform(0.0, 2 * math.pi)
    t = 120.0 + dt * np.arange(nt)
    A = A0 * np.sin(math.pi * t / 400.0) ** 2 * np.sin(om * t + cep)
    return A, 0.5 * (A + np.concatenate([[0.0], A[:-1]]))


def _inputs(case, seed):
    """The host data of a case, from the seed alone."""
    rs = np.random.RandomState(seed % (1 << 32))
    k = case["kind"]
    if k == "spectrum":
        nt, dt = case["nt"], 0.04
        t = dt * np.arange(nt)
        J = 1e-4 * sum(rs.standard_normal() * np.sin(w * t + rs.uniform(0, 6))
                       for w in rs.uniform(0.1, 1.5, 6))
        A = 0.05 * np.sin(math.pi * t / (dt * nt)) ** 2 * np.sin(rs.uniform(0.03, 0.1) * t)
        E = -np.diff(A, prepend=0.0) / dt
        return {"t": t, "J": J, "j0": float(J[0]), "E": E, "A": A, "dt": dt}
    ng, nb = case["ng"], case["nb"]
    acell, z, dt = CELLS[ng]
    s = {"acell": acell, "dt": dt, "ion": ([z], [1.0], [float(rs.uniform(0.0, 0.5))])}
    if k == "batch":
        nks = _nks(case)
        s["us"] = [_orbitals(rs, ng, nb, n, acell) for n in nks]
        f = [_field(rs, case["nt"], dt, "pulse") for _ in nks]
        s["A"], s["Aave"] = np.array([x[0] for x in f]), np.array([x[1] for x in f])
        return s
    nk = case["nk"]
    if k == "grad":
        s["us"] = [_orbitals(rs, ng, nb, nk, acell) for _ in range(case["ntraj"])]
        s["A"] = np.array([_field(rs, case["nt"], dt, "pulse")[0] for _ in s["us"]])
        return s
    s["u"] = _orbitals(rs, ng, nb, nk, acell)
    if k == "hpsi":
        s["w"], s["a"] = _orbitals(rs, ng, nb, nk, acell), float(rs.uniform(-0.3, 0.3))
    elif k == "step":
        s["a"], s["aave"] = float(rs.uniform(-0.3, 0.3)), float(rs.uniform(-0.3, 0.3))
    elif k == "rt":
        s["A"], s["Aave"] = _field(rs, case["nt"], dt, case["field"])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    k = case["kind"]
    if k == "spectrum":
        return s
    ng, nb, nbocc = case["ng"], case["nb"], case.get("nbocc", case["nb"])
    if k == "batch":
        nks = _nks(case)
        vion = {n: T.ion_potential(ng, n, s["acell"], *s["ion"]) for n in set(nks)}
        s["B"] = T.Batch(ng, nb, nbocc, s["acell"], s["dt"], nks, np.array([vion[n] for n in nks]))
        s["B"].upload(s["us"])
        if case["tune"]:
            s["B"].autotune(s["A"][:, :4], s["Aave"][:, :4])
        return s
    vion = T.ion_potential(ng, case["nk"], s["acell"], *s["ion"])
    s["G"] = T.TDHF(ng, case["nk"], nb, nbocc, s["acell"], s["dt"], vion)
    return s


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "hpsi":
        return s["G"].ubkwbk_hwbk(s["u"], s["w"], s["a"])
    if k == "step":
        return s["G"].RT_RK4_ubk(s["u"], s["aave"], s["a"])
    if k == "rt":
        return s["G"].RT_calculation(s["u"], s["A"], s["Aave"])
    if k == "batch":
        s["B"].upload(s["us"])
        e, n, j, i3 = s["B"].propagate(s["A"], s["Aave"])
        return s["B"].download(), e, n, j, i3
    if k == "grad":
        L, us, e, n, j = s["G"].fwd_batch(s["us"], s["A"], objective=case["objective"])
        g, gu = s["G"].bwd_batch()
        return L, us, e, n, j, g, gu
    if k == "gs":
        return s["G"].GS_calculation(s["u"], case["nscf"], case["ncg"])
    return T.fourier(s["t"], s["J"], s["j0"], s["E"], s["A"], s["dt"], case["nomega"], 2.0,
                     case["window"], s["dt"] * case["nt"])


# ---------------------------------------------------------------------------
# the same outputs in plain torch
# ---------------------------------------------------------------------------
class _Exact:
    """The equations in complex128: orbitals are (NK, NB, NG) tensors."""

    def __init__(self, ng, nk, nb, nbocc, acell, dt, ion):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.ng, self.nk, self.nb, self.nbocc = ng, nk, nb, nbocc
        self.acell, self.dt, self.dv, self.occ = acell, dt, acell / ng, 2.0 / nk
        b = 2 * math.pi / acell
        f64 = {"dtype": torch.float64, "device": self.dev}
        self.G = torch.tensor([(i if i < ng // 2 else i - ng) * b for i in range(ng)], **f64)
        self.k = torch.tensor([(-0.5 + (2 * i + 1) / (2 * nk)) * b for i in range(nk)], **f64)
        # soft Coulomb in k space: trapezoid over [0, NK acell) in steps of acell/NG/20
        dx, ns = acell / ng / 20.0, 0
        ns = int(math.ceil(nk * acell / dx)) - 2
        while ns * dx < nk * acell:
            ns += 1
        x = dx * torch.arange(ns + 1, **f64)
        wt = 2 * dx / torch.sqrt(x * x + 1.0)
        wt[0] *= 0.5
        wt[-1] *= 0.5
        d = torch.arange(-(nk - 1), nk, device=self.dev)
        i, j = torch.clamp(d, min=0), torch.clamp(-d, min=0)
        q = torch.cat([(self.G[None, :] + self.k[i][:, None] - self.k[j][:, None]).reshape(-1),
                       self.G])
        step = max(1, (1 << 26) // (ns + 1))
        v = torch.cat([(torch.cos(q[o:o + step, None] * x) * wt).sum(1)
                       for o in range(0, q.numel(), step)])
        self.vq, self.vg = v[:-ng].reshape(2 * nk - 1, ng), v[-ng:].clone()
        self.vg[0] = 0.0
        z, alpha, rion = ion
        r = acell * torch.arange(ng, **f64) / ng
        n = torch.arange(-4 * nk, 4 * nk + 1, **f64)
        self.vion = sum(-zi / torch.sqrt((r[:, None] - acell * ri - acell * n) ** 2 + ai * ai)
                        for zi, ai, ri in zip(z, alpha, rion)).sum(1)
        self.vion = self.vion - self.vion.max()
        # pairs of k-points in blocks of at most 2^26 grid values
        self.blk = max(1, (1 << 26) // (nk * nb * nbocc * ng))

    def get(self, u):
        return torch.tensor(np.ascontiguousarray(u.transpose(2, 1, 0)), device=self.dev)

    def put(self, u):
        return np.asfortranarray(u.detach().cpu().numpy().transpose(2, 1, 0))

    def rho(self, u):
        return self.occ * (u[:, :self.nbocc].abs() ** 2).sum((0, 1))

    def vh(self, rho):
        return torch.fft.ifft(self.vg * torch.fft.fft(rho.to(torch.complex128))).real

    def kin(self, w, A):
        q = self.G[None, :] + self.k[:, None] + A
        return torch.fft.ifft(0.5 * (q * q)[:, None, :] * torch.fft.fft(w))

    def fock(self, u, w):
        uo = u[:, :self.nbocc]

        def block(wb, uo, k0):
            ks = torch.arange(k0, k0 + wb.shape[0], device=self.dev)
            t = self.vq[ks[:, None] - torch.arange(self.nk, device=self.dev) + self.nk - 1]
            p = torch.fft.fft(wb[:, :, None, None, :] * uo.conj()[None, None])
            p = torch.fft.ifft(p * t[:, None, :, None, :])
            return (p * uo[None, None]).sum((2, 3)) * (-1.0 / self.nk)

        return torch.cat([block(w[o:o + self.blk], uo, o) for o in range(0, self.nk, self.blk)])

    def h(self, u, w, A):
        return self.kin(w, A) + (self.vh(self.rho(u)) + self.vion) * w + self.fock(u, w)

    def obs(self, u, A):
        """Etot, N, J."""
        uo, rho = u[:, :self.nbocc], self.rho(u)
        q = (self.G[None, :] + self.k[:, None] + A)[:, None, :]
        p2 = torch.fft.fft(uo).abs() ** 2 / self.ng
        ek = self.occ * self.dv * (0.5 * q * q * p2).sum()
        jj = -self.occ * self.dv / self.acell * (q * p2).sum()
        ex = 0.5 * self.occ * self.dv * (uo.conj() * self.fock(u, uo)).sum().real
        e = ek + self.dv * ((self.vion + 0.5 * self.vh(rho)) * rho).sum() + ex
        return torch.stack([e, self.dv * rho.sum(), jj])

    def f(self, u, A):
        return -1j * self.h(u, u, A)

    def step(self, u, Aave, A):
        dt = self.dt
        k1 = self.f(u, 2 * Aave - A)
        k2 = self.f(u + 0.5 * dt * k1, Aave)
        k3 = self.f(u + 0.5 * dt * k2, Aave)
        k4 = self.f(u + dt * k3, A)
        return u + (k1 + 2 * k2 + 2 * k3 + k4) * dt / 6


def _exact_rt(X, u, A, Aave):
    u = X.get(u)
    first, rows = X.obs(u, 0.0).cpu().numpy(), []
    for a, av in zip(A, Aave):
        u = X.step(u, float(av), float(a))
        rows.append(X.obs(u, float(a)))
    e, n, j = (r.copy() for r in torch.stack(rows).cpu().numpy().T)
    return X.put(u), e, n, j, first


def _exact_grad(X, u, A, objective):
    """Objective, final state, observables, dL/dA and dL/du0 of one pulse."""
    from torch.utils.checkpoint import checkpoint

    u0 = X.get(u).requires_grad_(True)
    a = torch.tensor(A, device=X.dev, requires_grad=True)
    prev = torch.cat([a.new_zeros(1), a[:-1]])
    u, rows, js = u0, [], []
    for n in range(a.numel()):
        u = checkpoint(X.step, u, 0.5 * (a[n] + prev[n]), a[n], use_reentrant=False)
        o = checkpoint(X.obs, u, a[n], use_reentrant=False)
        rows.append(o.detach())
        js.append(o)
    L = js[-1][0] if objective == "energy" else X.dt * sum(o[2] ** 2 for o in js)
    gu, ga = torch.autograd.grad(L, (u0, a))
    e, n, j = (r.copy() for r in torch.stack(rows).cpu().numpy().T)
    return float(L), X.put(u), e, n, j, ga.cpu().numpy(), X.put(gu)


def _exact_gs(X, u, nscf, ncg):
    """Energies, band energies and residuals; the orbitals' phases are free."""
    def orth(w):  # dv-orthonormal columns
        return torch.linalg.qr(w.transpose(1, 2))[0].transpose(1, 2) / math.sqrt(X.dv)

    def ritz(W, HW):
        s = torch.matmul(W.conj(), HW.transpose(1, 2).contiguous()) * X.dv
        _, v = torch.linalg.eigh(0.5 * (s + s.conj().transpose(1, 2)))
        return torch.matmul(v[:, :, :X.nb].transpose(1, 2).contiguous(), W)

    u = X.get(u)
    es = [X.obs(u, 0.0)[0]]
    for _ in range(nscf):
        u = orth(u)
        W = [u]
        for _ in range(1, ncg):
            W.append(X.h(u, W[-1], 0.0))
        W = orth(torch.cat(W, 1))
        HW = torch.cat([X.h(u, W[:, o:o + X.nb].contiguous(), 0.0)
                        for o in range(0, X.nb * ncg, X.nb)], 1)
        u = orth(ritz(W, HW))
        u = ritz(u, X.h(u, u, 0.0))
        es.append(X.obs(u, 0.0)[0])
    hu = X.h(u, u, 0.0)
    eps = (u.conj() * hu).sum(2).real * X.dv
    err = torch.sqrt((hu - eps[:, :, None] * u).abs().sum(2) * X.dv)
    return (None, torch.stack(es).cpu().numpy(), np.asfortranarray(eps.cpu().numpy().T),
            np.asfortranarray(err.cpu().numpy().T))


def _exact_spectrum(s, case):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t, J, E, A = (torch.tensor(s[n], device=dev) for n in ("t", "J", "E", "A"))
    nt, dt = case["nt"], s["dt"]
    if case["window"] == 0:
        r = t / t[-1]
        f = 1.0 - 3.0 * r * r + 2.0 * r * r * r
    else:
        f = torch.sin(math.pi * t / (dt * nt)) ** 2
    cols = torch.stack([f * (J - s["j0"]), f * E, f * A], 1)
    w = torch.arange(1, case["nomega"] + 1, dtype=torch.float64, device=dev) / case["nomega"] * 2.0
    out = []
    for o in range(0, w.numel(), 512):
        ph = w[o:o + 512, None] * t
        c = torch.stack([torch.matmul(torch.cos(ph), cols), torch.matmul(torch.sin(ph), cols)], 2)
        out.append(torch.cat([w[o:o + 512, None], dt * c.reshape(-1, 6)], 1))
    return torch.cat(out).cpu().numpy()


def exact(case, seed):
    s, k = _inputs(case, seed), case["kind"]
    if k == "spectrum":
        return _exact_spectrum(s, case)
    ng, nb, nbocc = case["ng"], case["nb"], case.get("nbocc", case["nb"])
    if k == "batch":
        nks, ntraj, nt = _nks(case), case["ntraj"], case["nt"]
        if 4 * nt * sum(_h_flops(ng, n, nb, nbocc) for n in nks) > 1.5e12:
            return None
        X = {n: _Exact(ng, n, nb, nbocc, s["acell"], s["dt"], s["ion"]) for n in set(nks)}
        rows = [_exact_rt(X[nks[t]], s["us"][t], s["A"][t], s["Aave"][t]) for t in range(ntraj)]
        return ([r[0] for r in rows],) + tuple(np.array([r[c] for r in rows]) for c in (1, 2, 3, 4))
    X = _Exact(ng, case["nk"], nb, nbocc, s["acell"], s["dt"], s["ion"])
    if k == "hpsi":
        return X.put(X.h(X.get(s["u"]), X.get(s["w"]), s["a"]))
    if k == "step":
        return X.put(X.step(X.get(s["u"]), s["aave"], s["a"]))
    if k == "rt":
        return _exact_rt(X, s["u"], s["A"], s["Aave"])
    if k == "gs":
        return _exact_gs(X, s["u"], case["nscf"], case["ncg"])
    rows = [_exact_grad(X, u, A, case["objective"]) for u, A in zip(s["us"], s["A"])]
    col = [[r[c] for r in rows] for c in range(7)]
    return (np.array(col[0]), col[1], np.array(col[2]), np.array(col[3]), np.array(col[4]),
            np.array(col[5]), col[6])
