"""The work that users of this package have it do, as cases that can be timed.

A case is a whole run as a caller's program makes it: initial state in, a
number of time steps, final state out (the solvers), or a run of pushes and
evaluations on device-resident data (the time sums, the exponential
accumulators).  Families and sizes are those of the package's workloads
(workloads.py, bench.py) and of its tests' small grids:

* lod2d      -- TGSolver, the 2D LOD solver, in every memory-term form
* mt1d       -- MT1DBatch, Caputo L1 (one problem up to batches)
* psi        -- MT1DBatch, psi-Caputo with nonlinear diffusivity and Picard
* ab1d       -- MT1DBatch, Atangana-Baleanu test problems, full history
* ab1d_series -- the same with the reference's series history
* timesum    -- TimeSum, the time sums of the 3D irrigation solver
* soe_step   -- SoeHistory, standalone exponential accumulators
"""
import math

import numpy as np
import torch

from theses_code_amd import _native as N
from theses_code_amd import workloads as W
from theses_code_amd.solvers import MT1DBatch, SoeHistory, TGSolver, TimeSum, coefs_advection

_PREC = {"f64": N.PREC_F64, "f32c": N.PREC_F32C, "mfma": N.PREC_MFMA_BF16, "soe": N.PREC_SOE}
_KERNEL = {"caputo": N.KERNEL_CAPUTO, "ab": N.KERNEL_AB}
TAU = 1e-3


def listed():
    lod = dict(family="lod2d", kernel="caputo", terms=0, soe_f32=False)
    return [
        # the smallest call: a unit-test sized grid, a few steps; launches and
        # latency are all of it
        dict(lod, name="lod2d_40x33_f64", form="f64", sN=40, M=33, steps=25, alpha=0.7),
        # one 1D problem over its whole run (a fitting driver's single particle)
        dict(name="mt1d_200", family="mt1d", nprob=1, Nmin=200, Nmax=200, steps=2000,
             precision="f64"),
        # the plain FP64 full history on the 512 x 512 convection-diffusion model
        dict(lod, name="lod2d_512_f64", form="f64", sN=513, M=513, steps=1000, alpha=0.7),
        # the 1024 x 1024 model in the three forms its precision study compares
        dict(lod, name="lod2d_1024_f32c", form="f32c", sN=1025, M=1025, steps=500, alpha=0.6),
        dict(lod, name="lod2d_1024_soe", form="soe", sN=1025, M=1025, steps=500, alpha=0.6,
             terms=32),
        dict(lod, name="lod2d_1024_mfma", form="mfma", sN=1025, M=1025, steps=2000, alpha=0.6),
        # one of the Atangana-Baleanu parameter sets: an odd side, no velocity,
        # slowly decaying weights (three BF16 parts)
        dict(lod, name="lod2d_1531_ab_mfma", form="mfma", kernel="ab", sN=1532, M=1532, steps=600,
             alpha=0.48),
        # thousands of uneven nonlinear moisture problems advanced together
        dict(name="psi_4096_f32c", family="psi", nprob=4096, Nmin=64, Nmax=1024, steps=400,
             precision="f32c", picard=3),
        # a batch of uneven Atangana-Baleanu test problems, full FP64 history
        dict(name="ab1d_1024", family="ab1d", nprob=1024, Nmin=64, Nmax=1024, steps=600),
        # the same test problems with the series history, all of one size
        dict(name="ab1d_series_1024", family="ab1d_series", nprob=1024, Nmin=100, Nmax=100,
             steps=600),
        # time sums on the 3D irrigation grid: a level pushed and summed per step
        dict(name="timesum_128x128x64", family="timesum", nodes=128 * 128 * 64, steps=200, alg=0,
             precision="f64", alpha=0.8, terms=0),
        # exponential accumulators at a large ragged node count, FP64 states
        dict(name="soe_step_20M", family="soe_step", nodes=20_000_003, modes=64, targets=1,
             f32=False, steps=4, alpha=0.8),
    ]


# ---------------------------------------------------------------- drawn cases
def _logint(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    """One more case of the listed families' ranges."""
    family = rng.choice(["lod2d"] * 5 + ["mt1d", "psi", "ab1d", "ab1d_series", "timesum",
                                         "soe_step"])
    if family == "lod2d":
        form = rng.choice(["f64", "f32c", "soe", "mfma"])
        kernel = rng.choice(["caputo", "caputo", "ab"])
        sN, M = _logint(rng, 24, 1540), _logint(rng, 24, 1540)
        nodes = (sN - 1) * (M - 1)
        most = {"f64": math.sqrt(2.6e11 / nodes), "f32c": math.sqrt(2.6e11 / nodes),
                "soe": 4.0e8 / nodes, "mfma": min(2.0e9 / nodes, math.sqrt(4e12 / nodes))}[form]
        steps = _logint(rng, 130 if form == "soe" else 20, min(1600, most))
        # the half-step Caputo scheme decays for orders above 0.55 only; the
        # Atangana-Baleanu split is stable over the parameter sets' range
        alpha = round(rng.uniform(0.6, 0.9) if kernel == "caputo" else rng.uniform(0.35, 0.85), 3)
        soe = form == "soe"
        return dict(family=family, form=form, kernel=kernel, sN=sN, M=M, steps=steps, alpha=alpha,
                    terms=(64 if kernel == "ab" else 32) if soe else 0,
                    soe_f32=bool(soe and kernel == "ab" and rng.random() < 0.5))
    if family == "mt1d":
        nprob = _logint(rng, 1, 1024)
        hi = rng.randint(50, 1024)
        lo = rng.choice([hi, max(3, hi // 8)])
        steps = _logint(rng, 60, min(2000, math.sqrt(2e11 / (nprob * 0.5 * (lo + hi)))))
        return dict(family=family, nprob=nprob, Nmin=lo, Nmax=hi, steps=steps,
                    precision=rng.choice(["f64", "f64", "f32c"]))
    if family == "psi":
        nprob = _logint(rng, 1, 4096)
        hi = rng.randint(128, 1024)
        return dict(family=family, nprob=nprob, Nmin=64, Nmax=hi, steps=_logint(rng, 40, 400),
                    precision=rng.choice(["f64", "f32c"]), picard=rng.randint(1, 3))
    if family == "ab1d":
        hi = rng.randint(128, 1024)
        return dict(family=family, nprob=_logint(rng, 1, 1024), Nmin=64, Nmax=hi,
                    steps=_logint(rng, 40, 600))
    if family == "ab1d_series":
        n = rng.randint(40, 300)
        return dict(family=family, nprob=_logint(rng, 1, 1024 * 100 // n), Nmin=n, Nmax=n,
                    steps=_logint(rng, 40, 600))
    if family == "timesum":
        alg = rng.choice([0, 0, 2])
        return dict(family=family, nodes=_logint(rng, 10_000, 1_048_576),
                    steps=_logint(rng, 30, 200), alg=alg,
                    precision="f64" if alg == 2 else rng.choice(["f64", "f32c"]),
                    alpha=round(rng.uniform(0.5, 0.9), 3), terms=16 if alg == 2 else 0)
    return dict(family=family, nodes=_logint(rng, 50_000, 20_000_000), modes=rng.randint(8, 64),
                targets=rng.randint(1, 2), f32=rng.random() < 0.3, steps=4,
                alpha=round(rng.uniform(0.5, 0.9), 3))


# ---------------------------------------------------------------- inputs
_ctx = None


def _context():
    """The program's one context (device 0)."""
    global _ctx
    if _ctx is None:
        _ctx = N.Context(0)
    return _ctx


class _View:
    """A solver's device buffer as torch takes one."""

    def __init__(self, d, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(d.n,), typestr="<f8", data=(d.ptr, False),
                                             version=3)


def _tensor(d, owner):
    t = torch.as_tensor(_View(d, owner), device="cuda")
    t.owner = owner  # the buffer goes with its solver, so the solver stays while the tensor does
    return t


class _State:
    """What a caller's program holds between calls; device arrays that it
    allocated go when it does."""

    def __init__(self, case, **kw):
        self.case = case
        self.arrays = []
        self.__dict__.update(kw)

    def device(self, a):
        d = N.DeviceArray.from_host(_context(), a)
        self.arrays.append(d)
        return d

    def __del__(self):
        for d in self.arrays:
            d.free()


def _modes_field(rng, ny, nx, h, corr, modes=24):
    """A smooth random field: random Fourier modes with a Gaussian spectrum."""
    k = rng.normal(size=(2, modes)) * (math.sqrt(2.0) / corr)
    ph = rng.uniform(0, 2 * math.pi, modes)
    ax = np.exp(1j * np.outer(np.arange(nx) * h, k[0]))
    ay = np.exp(1j * (np.outer(np.arange(ny) * h, k[1]) + ph))
    return np.real(ay @ ax.T) * math.sqrt(2.0 / modes)


def _lod_inputs(c, seed):
    """(coefs, C0): advection by the curl of a smooth stream function with a
    sum of blobs, or (Atangana-Baleanu sets) pure diffusion of a smooth field."""
    rng = np.random.default_rng(seed)
    nx, ny = c["sN"] + 2, c["M"] + 2
    h = 1.0 / max(c["sN"], c["M"])
    D = 1e-3
    if c["kernel"] == "ab":
        zero = np.zeros((ny, nx))
        return coefs_advection(zero, zero, D, h), 0.5 + 0.1 * _modes_field(rng, ny, nx, h, 0.1)
    psi = _modes_field(rng, ny, nx, h, 0.1)
    vx = np.gradient(psi, h, axis=0)
    vy = -np.gradient(psi, h, axis=1)
    s = 0.1 / np.max(np.hypot(vx, vy))
    x, y = np.arange(nx) * h, np.arange(ny) * h
    a, cx, cy = rng.uniform(0, 1, (3, 8))
    gx = np.exp(-(x[:, None] - cx) ** 2 / (2 * 0.05 ** 2))
    gy = np.exp(-(y[:, None] - cy) ** 2 / (2 * 0.05 ** 2))
    return coefs_advection(vx * s, vy * s, D, h), (gy * a) @ gx.T


def _sizes(c):
    """The problems' interval counts: part of the case, the same for every seed."""
    rng = np.random.default_rng([c["nprob"], c["Nmin"], c["Nmax"]])
    return rng.integers(c["Nmin"], c["Nmax"] + 1, c["nprob"])


def _mt1d_inputs(c, seed):
    """Caputo diffusion problems as the 200-interval workload, fixed ends."""
    rng = np.random.default_rng(seed)
    probs, U0 = [], []
    single = c["nprob"] == 1
    for n in _sizes(c).tolist():
        x = np.arange(n + 2) / n
        top, bot = (0.0, 0.0) if single else rng.uniform(0, 0.2, 2)
        u = np.sin(math.pi * x) + 0.01 * rng.normal(size=n + 2)
        u[0], u[n], u[n + 1] = top, bot, bot
        probs.append(dict(N=n, L=1.0, alpha=0.8 if single else float(rng.uniform(0.5, 0.95)),
                          form=N.FORM_CONST, D=1e-3 if single else float(rng.uniform(1e-4, 1e-2)),
                          top=N.TOP_DIRICHLET, top_val=float(top), bottom_cond=1,
                          Hbottom=float(bot)))
        U0.append(u)
    return probs, U0


def _psi_inputs(c, seed):
    """Moisture problems k(u) = k0 exp(b u), psi(t) = t^beta, wet top, flux bottom."""
    rng = np.random.default_rng(seed)
    probs, U0 = [], []
    for n in _sizes(c).tolist():
        probs.append(dict(N=n, L=1.0, alpha=float(rng.uniform(0.5, 0.99)),
                          beta=float(rng.uniform(0.5, 1.5)), form=N.FORM_KEXP,
                          k0=float(rng.uniform(1e-4, 1e-2)), b=float(rng.uniform(0.0, 3.0)),
                          top=N.TOP_DIRICHLET, top_val=0.4, bottom_cond=0))
        u = rng.uniform(0.1, 0.4, n + 2)
        u[0], u[n + 1] = 0.4, u[n]
        U0.append(u)
    return probs, U0


def _ab1d_inputs(c, seed, series):
    """Manufactured Atangana-Baleanu solutions started from a perturbed field."""
    rng = np.random.default_rng(seed)
    orders = np.round(np.arange(0.9, 0.05, -0.1), 1) if series else np.linspace(0.3, 0.9, 16)
    cfg = W.AB1D_SERIES_WORKLOAD if series else W.AB1D_WORKLOAD
    probs, U0 = [], []
    for q, n in enumerate(_sizes(c).tolist()):
        probs.append(dict(N=n, alpha=float(orders[q % orders.size]), src=int(rng.integers(0, 3)),
                          ab_maxl=cfg["maxl"], ab_maxkiter=cfg["maxkiter"], ab_eps=cfg["eps"],
                          ab_series=int(series)))
        u = 0.1 * np.sin(math.pi * np.arange(n + 2) / n) * rng.uniform(0.5, 1.0)
        u[0] = u[n] = u[n + 1] = 0.0
        U0.append(u)
    return probs, U0


def _batch_args(c, seed):
    f = c["family"]
    if f == "mt1d":
        return _mt1d_inputs(c, seed), TAU, dict(kind=N.MT_L1, precision=_PREC[c["precision"]])
    if f == "psi":
        return _psi_inputs(c, seed), TAU, dict(kind=N.MT_PSI, precision=_PREC[c["precision"]],
                                               picard=c["picard"])
    cfg = W.AB1D_SERIES_WORKLOAD if f == "ab1d_series" else W.AB1D_WORKLOAD
    return _ab1d_inputs(c, seed, f == "ab1d_series"), cfg["tau"], dict(kind=N.MT_AB)


def _levels(c, seed):
    """Eight distinct time levels, pushed in turn (smooth in time)."""
    rng = np.random.default_rng(seed)
    base, rate = rng.uniform(-1, 1, (2, c["nodes"]))
    return [base + rate * math.sqrt(k + 1.0) for k in range(8)]


def _timesum_weights(c):
    """Per step: the evaluation's arguments, as the 3D solver's caller has them."""
    tau, K, al = W.TIMESUM3D_WORKLOAD["tau"], c["steps"], c["alpha"]
    T = np.arange(K + 2) * tau
    if c["alg"] == 2:
        j = np.arange(c["terms"])
        return [dict(coefs=(T[k + 1] ** (j + 1) - T[k] ** (j + 1)) / ((j + 1) * T[k + 1] ** (j + 1)),
                     gtj=T[k + 2], gt=T[k + 1], alpha=al, tau_n=tau) for k in range(K)]
    taus = np.full(K + 1, tau)
    return [dict(kb_3_cache=W.caputo_interval_weights(T[:k + 2], T[k + 1], al), tau=taus)
            for k in range(K)]


def _soe_coefs(c):
    """Decays and per-target coefficients on logarithmically spaced rates."""
    L = c["modes"]
    r = np.logspace(-4, 0.5, L)
    q = np.exp(-r)
    t0 = r ** c["alpha"] / L
    return q, np.stack([t0, t0 * np.exp(-0.5 * r)])[:c["targets"]]


def prepare(case, seed):
    c, ctx = dict(case), _context()
    f = c["family"]
    if f == "lod2d":
        coefs, C0 = _lod_inputs(c, seed)
        kw = {}
        if c["form"] == "soe":
            kw.update(soe_terms=c["terms"], soe_f32=c["soe_f32"])
        s = TGSolver(ctx, c["sN"], c["M"], c["alpha"], TAU, 1.0, coefs, C0, capacity=c["steps"],
                     C1=0.0 if c["kernel"] == "caputo" else 0.5, precision=_PREC[c["form"]],
                     kernel=_KERNEL[c["kernel"]], ab_exact=c["kernel"] == "ab", **kw)
        return _State(c, solver=s, C0=C0)
    if f in ("mt1d", "psi", "ab1d", "ab1d_series"):
        (probs, U0), tau, kw = _batch_args(c, seed)
        return _State(c, solver=MT1DBatch(ctx, probs, tau, c["steps"], U0, **kw), U0=U0)
    if f == "timesum":
        s = _State(c, solver=TimeSum(ctx, c["nodes"], sum_alg=c["alg"],
                                     sum_param=float(c["terms"]), capacity=c["steps"] + 1,
                                     precision=_PREC[c["precision"]]), args=_timesum_weights(c))
        s.levels = [s.device(a) for a in _levels(c, seed)]
        return s
    q, co = _soe_coefs(c)
    s = _State(c, solver=SoeHistory(ctx, c["nodes"], c["modes"], c["targets"], f32=c["f32"]), q=q,
               co=co)
    rng = np.random.default_rng(seed)
    s.incr = [s.device(rng.random(c["nodes"]) * 2 - 1) for _ in range(2)]
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    c, s = state.case, state.solver
    f = c["family"]
    if f == "lod2d":
        s.set_state(state.C0)
        s.calc_step(c["steps"])
        return s.b_C
    if f in ("mt1d", "psi"):
        s.set_state(state.U0)
        s.calc_step(c["steps"])
        return s.state()[0].base  # the packed states that the list's views share
    if f in ("ab1d", "ab1d_series"):
        s.set_state(state.U0)
        s.calc_step(c["steps"])
        return s.state()[0].base, s.ab_error()
    if f == "timesum":
        s.clear()
        s.push(state.levels[0])
        for k in range(c["steps"]):
            s.push(state.levels[(k + 1) % len(state.levels)])
            S = s.eval_device(**state.args[k])
        return _tensor(S, s)
    s.clear()
    for k in range(c["steps"]):
        out = s.step_device(state.incr[k % len(state.incr)], state.q, state.co)
    return _tensor(out, s)


# ---------------------------------------------------------------- work
def work(case):
    c, f, T = case, case["family"], case["steps"]
    if f == "lod2d":
        nodes = (c["sN"] + 2) * (c["M"] + 2)
        # two targets per node and step: a term per past step, or per mode its
        # update and two terms; two sweeps of about 16 operations
        hist = 6.0 * c["terms"] if c["form"] == "soe" else 2.0 * (T - 1)
        return dict(bytes=nodes * 8.0 * 6, flops=nodes * T * (hist + 32.0))
    if f in ("mt1d", "psi", "ab1d", "ab1d_series"):
        nodes = c["nprob"] * (0.5 * (c["Nmin"] + c["Nmax"]) + 2)
        hist = 50 * 4.0 if f == "ab1d_series" else T - 1.0
        return dict(bytes=nodes * 8.0 * 2, flops=nodes * T * (hist + 30.0 * c.get("picard", 1)))
    if f == "timesum":
        # every level is summed at every step: the sums' weights come with the call
        if c["alg"] == 2:
            return dict(bytes=c["nodes"] * 8.0 * T * (2 * c["terms"] + 2),
                        flops=c["nodes"] * 4.0 * T * c["terms"])
        esz = 4.0 if c["precision"] == "f32c" else 8.0
        return dict(bytes=c["nodes"] * (esz * T * (T + 1) / 2 + 16.0 * T),
                    flops=c["nodes"] * 1.0 * T * (T + 1))
    esz = 4.0 if c["f32"] else 8.0
    return dict(bytes=c["nodes"] * T * (2 * esz * c["modes"] + 8.0 + 8.0 * c["targets"]),
                flops=c["nodes"] * T * c["modes"] * 2.0 * (1 + c["targets"]))


# ---------------------------------------------------------------- 64-bit values
def _gpu(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


class _Lines:
    """x_{i-1} a - R x_i + b x_{i+1} = om along `dim` of every line, by cyclic
    reduction with the matrices' part done once."""

    def __init__(self, a, R, b, dim):
        self.dim, self.levels = dim, []
        n = a.shape[dim]
        A, B, self.inv0 = a / R, b / R, -1.0 / R
        s = 1
        while s < n:
            den = 1.0 - A * self._from(B, -s) - B * self._from(A, s)
            self.levels.append((s, A / den, B / den, 1.0 / den))
            A, B = A * self._from(A, -s) / den, B * self._from(B, s) / den
            s *= 2

    def _from(self, x, s):
        """y_i = x_{i+s}, 0 outside"""
        y, n = torch.zeros_like(x), x.shape[self.dim]
        if s > 0:
            y.narrow(self.dim, 0, n - s).copy_(x.narrow(self.dim, s, n - s))
        else:
            y.narrow(self.dim, -s, n + s).copy_(x.narrow(self.dim, 0, n + s))
        return y

    def solve(self, om):
        d, k = om * self.inv0, self.dim
        n = d.shape[k]
        for s, A, B, inv in self.levels:
            e = d * inv
            e.narrow(k, s, n - s).addcmul_(A.narrow(k, s, n - s), d.narrow(k, 0, n - s))
            e.narrow(k, 0, n - s).addcmul_(B.narrow(k, 0, n - s), d.narrow(k, s, n - s))
            d = e
        return d


class _History:
    """sum_s w_t[n - s - 1] Delta_s for targets t, blocks of 64 steps at a time."""

    def __init__(self, w, steps, nodes):
        self.w, self.B, self.n = w, 64, 0
        self.d = torch.empty((steps, nodes), dtype=torch.float64, device="cuda")

    def sums(self):
        n, nt = self.n, self.w.shape[0]
        n0 = n - n % self.B
        if n == n0 and n > 0:  # the settled part for the block's steps
            lag = n + torch.arange(self.B, device="cuda")[:, None] - \
                torch.arange(n, device="cuda")[None, :]
            lag = torch.clamp(lag, max=self.w.shape[1])
            self.far = (self.w[:, lag - 1].reshape(nt * self.B, n) @ self.d[:n]).reshape(
                nt, self.B, -1)
        s = self.far[:, n - n0].clone() if n0 > 0 else torch.zeros(
            (nt, self.d.shape[1]), dtype=torch.float64, device="cuda")
        if n > n0:
            s += self.w[:, :n - n0].flip(1) @ self.d[n0:n]
        return s

    def push(self, x):
        self.d[self.n] = x.reshape(-1)
        self.n += 1


def _ab_integrals(a, tau, D):
    """integral of E_a(-a/(1-a) u^a) over [(d-1) tau, d tau], d = 1..D, from the
    spectral form of the kernel by the trapezoid rule in log r."""
    lam, sa, ca = a / (1 - a), math.sin(math.pi * a), math.cos(math.pi * a)
    x = torch.arange(-60.0 / a, 90.0 / a, 0.02, dtype=torch.float64, device="cuda")
    r = torch.exp(x)
    # mu(r) dr / r = [lam sa / pi] / (r^a + 2 lam ca + lam^2 r^-a) dx / r * r^0
    mu = lam * sa / math.pi / (torch.exp(a * x) + 2 * lam * ca + lam * lam * torch.exp(-a * x)) * 0.02
    base = mu * -torch.expm1(-r * tau) / r
    return torch.stack([(base * torch.exp(-r * (d * tau))).sum() for d in range(D)])


def _lod_exact(c, seed):
    coefs, C0 = _lod_inputs(c, seed)
    sN, M, T, al = c["sN"], c["M"], c["steps"], c["alpha"]
    rA, rB, cA, cB = [_gpu(np.broadcast_to(v, C0.shape))[1:M, 1:sN].clone() for v in coefs]
    C = _gpu(C0)
    sg, caputo = 1.0 / TAU, c["kernel"] == "caputo"
    if caputo:
        k = torch.arange(1, T + 1, dtype=torch.float64, device="cuda")
        g = TAU ** (1 - al) / math.gamma(2 - al)

        def kb(d, l):
            return -g * d ** (1 - al) * torch.expm1((1 - al) * torch.log1p(-l / d))
        w = torch.stack([kb(k + 0.5, 1.0), kb(k + 1.0, 1.0)])
        k0 = g * 0.5 ** (1 - al)
        kch = g * (1.0 - 0.5 ** (1 - al))
        C1 = 0.0
    else:
        I = _ab_integrals(al, TAU, T + 1) / (1 - al)
        w, k0, kch, C1 = (0.5 * I[1:]).expand(2, -1).contiguous(), float(I[0]), 0.0, 0.5
    Rr, Rc = sg * k0 + rA + rB, sg * k0 + cA + cB
    left = rA[:, 0].clone() * C1  # Dirichlet C1 at i = 0
    rA[:, 0] = 0.0
    Rr[:, -1] -= rB[:, -1]  # zero gradient at i = sN and at both column ends
    rB[:, -1] = 0.0
    Rc[0] -= cA[0]
    cA[0] = 0.0
    Rc[-1] -= cB[-1]
    cB[-1] = 0.0
    rows, cols = _Lines(rA, Rr, rB, 1), _Lines(cA, Rc, cB, 0)
    hist = _History(w, T, (sN - 1) * (M - 1))
    for _ in range(T):
        prev = C[1:M, 1:sN].clone()
        s = hist.sums().reshape(2, M - 1, sN - 1)
        om = -sg * k0 * prev + sg * s[0]
        om[:, 0] -= left
        u = rows.solve(om)
        C[1:M, 1:sN] = u
        C[1:M, 0] = C1
        C[1:M, sN], C[1:M, sN + 1] = u[:, -1], u[:, -1]
        om = -sg * k0 * u + sg * (s[1] + kch * (prev - u))
        u = cols.solve(om)
        C[1:M, 1:sN] = u
        C[0, 1:sN], C[M, 1:sN], C[M + 1, 1:sN] = u[0], u[-1], u[-1]
        hist.push(u - prev)
    return C


def _mt1d_exact(c, seed):
    probs, U0 = _mt1d_inputs(c, seed)
    T, P, n = c["steps"], len(probs), c["Nmax"] - 1

    def col(f):
        return _gpu([f(p) for p in probs])[:, None]
    al = col(lambda p: p["alpha"])
    Nn = col(lambda p: p["N"])
    Da = col(lambda p: TAU ** -p["alpha"] / math.gamma(2 - p["alpha"]))
    g = col(lambda p: p["D"]) * Nn * Nn
    top, bot = col(lambda p: p["top_val"]), col(lambda p: p["Hbottom"])
    i = torch.arange(n, dtype=torch.float64, device="cuda")[None]
    real, first, last = i < Nn - 1, i == 0, i == Nn - 2
    a = torch.where(real & ~first, g, 0.0 * g)
    b = torch.where(real & ~last, g, 0.0 * g)
    R = torch.where(real, 2 * g + Da, 1.0 + 0.0 * g)
    lines = _Lines(a, R, b, 1)
    ends = torch.where(first, g * top, 0.0 * g) + torch.where(last & real, g * bot, 0.0 * g)
    u = torch.zeros((P, n), dtype=torch.float64, device="cuda")
    for q, x in enumerate(U0):
        u[q, :probs[q]["N"] - 1] = _gpu(x[1:probs[q]["N"]])
    # lag l + 1 of the stored increments weighs (l+2)^(1-a) - (l+1)^(1-a); the
    # first two steps' increments are not stored
    l = torch.arange(T, dtype=torch.float64, device="cuda")[None]
    w = (l + 2) ** (1 - al) - (l + 1) ** (1 - al)
    d = torch.zeros((P, T, n), dtype=torch.float64, device="cuda")
    depth = 0
    for k in range(1, T + 1):
        om = -Da * u - ends
        if depth:
            om = om + Da * torch.matmul(w[:, None, :depth].flip(2), d[:, :depth])[:, 0]
        v = torch.where(real, lines.solve(om), 0.0 * u)
        if k >= 3:
            d[:, depth] = v - u
            depth += 1
        u = v
    out = []
    for q, p in enumerate(probs):
        m = p["N"]
        out.append(np.concatenate([[p["top_val"]], u[q, :m - 1].cpu().numpy(),
                                   [p["Hbottom"], p["Hbottom"]]]))
    return np.concatenate(out)


def _timesum_exact(c, seed):
    lev = [_gpu(a) for a in _levels(c, seed)]
    K, args = c["steps"], _timesum_weights(c)
    diff = [lev[(k + 1) % 8] - lev[k % 8] for k in range(8)]
    S = torch.zeros(c["nodes"], dtype=torch.float64, device="cuda")
    if c["alg"] == 2:
        m = torch.zeros((c["terms"], c["nodes"]), dtype=torch.float64, device="cuda")
        for k in range(K):
            A = args[k]
            for j in range(c["terms"]):
                m[j] += A["gt"] ** (j + 1) * A["coefs"][j] * diff[k % 8]
        v = A["gtj"] ** -c["alpha"]
        for j in range(c["terms"]):
            S += v * m[j]
            v *= (c["alpha"] + j) / ((j + 1) * A["gtj"])
        return S / A["tau_n"]
    A = args[K - 1]
    for k in range(K):
        S += float(A["kb_3_cache"][k] / A["tau"][k]) * diff[k % 8]
    return S


def _soe_exact(c, seed):
    rng = np.random.default_rng(seed)
    inc = [_gpu(rng.random(c["nodes"]) * 2 - 1) for _ in range(2)]
    q, co = _soe_coefs(c)
    out = torch.zeros((c["targets"], c["nodes"]), dtype=torch.float64, device="cuda")
    for k in range(c["steps"]):  # an increment k steps before the last one
        for t in range(c["targets"]):
            out[t] += float(np.sum(co[t] * q ** k)) * inc[(c["steps"] - 1 - k) % 2]
    return out.reshape(-1)


def exact(case, seed):
    """What run() returns, in 64 bits.  None for the psi and Atangana-Baleanu
    batches: their weights are the reference's series and quadratures cut at
    its own tolerances, so no independent 64-bit value exists."""
    f = case["family"]
    if f == "lod2d":
        return _lod_exact(case, seed)
    if f == "mt1d":
        nodes = case["nprob"] * case["Nmax"]
        return _mt1d_exact(case, seed) if nodes * case["steps"] ** 2 < 3e11 else None
    if f == "timesum":
        return _timesum_exact(case, seed)
    if f == "soe_step":
        return _soe_exact(case, seed)
    return None
