"""The work that is timed: what programs have this package do, through its
public entry points.

Every state is in the reference layout X[f*N + k*nr + i] (f = psi, T, S;
N = N_fm*nr, nr = N_r - 1), float64.  A case names its ``kind``:

  step        Plan.step on a batch, eager launches, out of place; with
              ``monitor`` the diagnostics of the result behind it
  graph       Plan.graph: nsteps in-place steps of a batch, one graph replay
  sweep       batching.Sweep: instances of mixed sizes and parameters in one
              graph replay
  linearised  Plan.step_linearized on a batch (J v of the Newton solves)
  newton      newton.Krylov.newton, one steady state
  newtons     newton.NewtonBatch.solve, several steady states of one class
  time_loop   the drop-in Main._Time_Step on host arrays: step, diagnostics
              and checkpoints
  transforms  sddc_transform, the four transforms of a block of rows

``exact`` restates the method in plain NumPy (float64): operators, transforms
as dense matrices, mode-by-mode back substitution, GMRES for the Newton
solves.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

from spectraldoublediffusiveconvection_amd import _lib, autotune, batching, device, newton
from spectraldoublediffusiveconvection_amd.dropin import Main

# parameters of the benchmark and of the thin-gap steady convection case
RUN = dict(d=0.35, Pr=1.0, Tau=1.0 / 15.0, dt=5e-3, Ra_s=500.0, Ra_lo=2500.0, Ra_hi=3000.0)
THIN = dict(d=0.353, Pr=1.0, Tau=1.0, dt=1.0, Ra=2360.0, Ra_s=0.0)
STEADY = os.path.join("tests", "golden", "convecting_thin_gap.npz")   # at N_fm = 48, N_r = 24


def listed():
    return [
        # one step of the smallest class a parameter study starts with:
        # launches and latency
        dict(name="step_one_small", kind="step", N_fm=64, N_r=20, batch=1, nsteps=1,
             precision="fp64", symmetric=False, monitor=False, tuned=False),
        # one plain float64 integration at production resolution
        dict(name="run_one_full", kind="step", N_fm=512, N_r=40, batch=1, nsteps=20,
             precision="fp64", symmetric=False, monitor=False, tuned=False),
        # a short run of an odd size, equatorially symmetric, watched: what a
        # resolution study does between the powers of two
        dict(name="run_ragged_watched", kind="step", N_fm=90, N_r=25, batch=13, nsteps=10,
             precision="fp64", symmetric=True, monitor=True, tuned=False),
        # a medium mixed-precision batch on a grid that is no multiple of 64
        dict(name="run_odd_mixed", kind="step", N_fm=300, N_r=48, batch=24, nsteps=5,
             precision="mixed", symmetric=False, monitor=True, tuned=False),
        # the headline batch: 256 mixed-precision instances, graph replay
        dict(name="graph_full_mixed", kind="graph", N_fm=512, N_r=40, batch=256, nsteps=20,
             precision="mixed", symmetric=False, tuned=True),
        # a medium float64 batch, graph replay
        dict(name="graph_mid_fp64", kind="graph", N_fm=256, N_r=30, batch=64, nsteps=10,
             precision="fp64", symmetric=False, tuned=True),
        # a sweep over resolutions and Rayleigh numbers in one graph
        dict(name="sweep_mixed_sizes", kind="sweep", instances=96, nsteps=10,
             precision="mixed"),
        # one J v of a Newton solve at production resolution
        dict(name="linearised_full", kind="linearised", N_fm=512, N_r=40, batch=1,
             precision="fp64", symmetric=False),
        # one steady state by Newton-Krylov (the drop-in's _Newton)
        dict(name="newton_small", kind="newton", N_fm=64, N_r=24, restart=100),
        # the serving engine's Newton worker: a batch of steady states
        dict(name="newtons_batch", kind="newtons", N_fm=96, N_r=24, batch=6, restart=100),
        # the reference's driver: a numpy state in, a numpy state out, with
        # diagnostics every step and its checkpoint file
        dict(name="time_loop_mid", kind="time_loop", N_fm=128, N_r=30, nsteps=20,
             symmetric=False),
        # the transforms of a block of rows at the 3/2-dealiased length
        dict(name="transforms_block", kind="transforms", N_fm=512, rows=2496),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def even(lo, hi):
        return 2 * int(round(log(lo, hi) / 2))

    kind = rng.choice(["step", "step", "step", "graph", "graph", "sweep", "linearised", "newton",
                       "newtons", "time_loop", "transforms"])
    N_fm, N_r = even(16, 512), rng.randint(10, 48)
    if rng.random() < 0.3:
        N_fm, N_r = rng.choice([64, 128, 256, 512]), rng.choice([20, 30, 40])
    per = N_fm * (N_r - 1)
    if kind in ("step", "graph"):
        batch = int(round(log(1, 256)))
        batch = max(1, min(batch, 5000000 // per))
        nsteps = int(round(log(1, 20)))
        nsteps = max(1, min(nsteps, 60000000 // (per * batch)))
        case = dict(kind=kind, N_fm=N_fm, N_r=N_r, batch=batch, nsteps=nsteps,
                    precision=rng.choice(["fp64", "mixed"]), symmetric=rng.random() < 0.3,
                    tuned=rng.random() < 0.5)
        if kind == "step":
            case["monitor"] = rng.random() < 0.5
        return case
    if kind == "sweep":
        return dict(kind=kind, instances=int(round(log(12, 128))), nsteps=rng.randint(2, 10),
                    precision=rng.choice(["fp64", "mixed"]))
    if kind == "linearised":
        return dict(kind=kind, N_fm=N_fm, N_r=N_r, batch=max(1, int(round(log(1, 16)))),
                    precision="fp64", symmetric=rng.random() < 0.3)
    if kind == "newton":
        return dict(kind=kind, N_fm=even(48, 128), N_r=rng.randint(22, 30), restart=100)
    if kind == "newtons":
        return dict(kind=kind, N_fm=even(48, 96), N_r=rng.randint(22, 26),
                    batch=rng.randint(2, 8), restart=100)
    if kind == "time_loop":
        return dict(kind=kind, N_fm=N_fm, N_r=N_r, nsteps=rng.randint(3, 20),
                    symmetric=rng.random() < 0.5)
    return dict(kind=kind, N_fm=N_fm, rows=int(round(log(1, 4000))))


# ------------------------------------------------------------------- inputs
def _states(batch, n3, seed):
    """Seeded normal states of norm 1e-3: the start of a run."""
    X = np.random.default_rng(seed).standard_normal((batch, n3))
    return 1e-3 * X / np.linalg.norm(X, axis=1, keepdims=True)


def _run_inputs(case, seed):
    n3 = 3 * case["N_fm"] * (case["N_r"] - 1)
    X = _states(case["batch"], n3, seed)
    Ra = np.random.default_rng(seed + 1000003).uniform(RUN["Ra_lo"], RUN["Ra_hi"], case["batch"])
    return X, Ra


def _linearised_inputs(case, seed):
    """A smooth state of order one (convecting flow) and a Krylov vector."""
    rng = np.random.default_rng(seed)
    K, nr, B = case["N_fm"], case["N_r"] - 1, case["batch"]
    X = 0.1 * rng.standard_normal((B, 3, K, nr)) * np.exp(-np.arange(K) / 10.0)[:, None]
    v = rng.standard_normal((B, 3 * K * nr))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    return X.reshape(B, -1), v, rng.uniform(RUN["Ra_lo"], RUN["Ra_hi"], B)


def _steady(K, Nr):
    """The committed steady thin-gap state moved to (K, Nr): barycentric
    interpolation in r on the Chebyshev points, zero padding in theta."""
    X = np.load(STEADY)["X24"].reshape(3, 48, 23)
    x0 = np.cos(np.pi * np.arange(25) / 24)
    x1 = np.cos(np.pi * np.arange(1, Nr) / Nr)
    w = (-1.0) ** np.arange(25)
    w[[0, -1]] *= 0.5
    diff = x1[:, None] - x0[None, :]
    same = np.abs(diff) < 1e-14
    C = w / np.where(same, 1.0, diff)
    C /= C.sum(axis=1, keepdims=True)
    C[same.any(axis=1)] = 0.0
    C[same] = 1.0
    out = np.zeros((3, K, Nr - 1))
    k = min(K, 48)
    out[:, :k] = X[:, :k] @ C[:, 1:-1].T
    return out


def _newton_inputs(case, seed):
    """Starts within 0.1% of the steady state, Ra_T within 0.02% of 2360 (close
    to onset, as the serving stream's Newton jobs)."""
    B = case.get("batch", 1)
    rng = np.random.default_rng(seed)
    base = _steady(case["N_fm"], case["N_r"])
    shape = (B,) + base.shape
    X = base * (1.0 + 1e-3 * rng.uniform(-1, 1, shape))
    Ra = THIN["Ra"] * (1.0 + 2e-4 * rng.uniform(-1, 1, B))
    return X.reshape(B, -1), Ra


def _sweep_inputs(case, seed):
    """Instances dealt over the sweep's twelve resolutions in turn."""
    rng = np.random.default_rng(seed)
    sizes = [(K, r) for r in (20, 30, 40) for K in (64, 128, 256, 512)]
    out = []
    for i in range(case["instances"]):
        K, Nr = sizes[i % len(sizes)]
        out.append(dict(N_fm=K, N_r=Nr, d=RUN["d"], dt=RUN["dt"], Pr=RUN["Pr"], Tau=RUN["Tau"],
                        Ra=float(rng.uniform(RUN["Ra_lo"], RUN["Ra_hi"])),
                        Ra_s=float(rng.choice((300.0, 500.0))),
                        X0=_states(1, 3 * K * (Nr - 1), seed + 7919 * i)[0]))
    return out


def _transform_inputs(case, seed):
    rng = np.random.default_rng(seed)
    K, M = case["N_fm"], 3 * case["N_fm"] // 2
    a = rng.standard_normal((case["rows"], K)) * np.exp(-np.arange(K) / (K / 6.0))
    return a, rng.standard_normal((case["rows"], M))


def _time_loop_inputs(case, seed):
    X = _states(1, 3 * case["N_fm"] * (case["N_r"] - 1), seed)[0]
    return X, float(np.random.default_rng(seed + 1000003).uniform(RUN["Ra_lo"], RUN["Ra_hi"]))


def _dev(a):
    return torch.as_tensor(a, device="cuda")


def _plan(case, dt, p, batch=1, symmetric=None):
    tuning = None
    if case.get("tuned"):
        tuning = autotune.TuningTable().lookup((case["N_fm"], case["N_r"]), batch,
                                               case["precision"])
    return device.Plan.build(case["N_fm"], case["N_r"], p["d"], dt, p["Pr"], p["Tau"],
                             symmetric=case["symmetric"] if symmetric is None else symmetric,
                             precision=case.get("precision", "fp64"), max_batch=batch,
                             tuning=tuning)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case)
    if kind in ("step", "graph"):
        X, Ra = _run_inputs(case, seed)
        s["plan"] = _plan(case, RUN["dt"], RUN, case["batch"])
        s["X"], s["Ra"] = _dev(X), _dev(Ra)
        s["Ra_s"] = _dev(np.full(case["batch"], RUN["Ra_s"]))
        if kind == "step":
            s["out"] = torch.empty_like(s["X"])
        else:
            s["graph"] = s["plan"].graph(s["X"], s["Ra"], s["Ra_s"], nsteps=case["nsteps"])
    elif kind == "sweep":
        s["sweep"] = batching.Sweep(_sweep_inputs(case, seed), precision=case["precision"],
                                    tuning_table=autotune.TuningTable())
        s["graph"] = s["sweep"].graph(nsteps=case["nsteps"])
    elif kind == "linearised":
        X, v, Ra = _linearised_inputs(case, seed)
        s["plan"] = _plan(case, 1.0, RUN, case["batch"])
        s["X"], s["v"], s["Ra"] = _dev(X), _dev(v), _dev(Ra)
        s["Ra_s"] = _dev(np.full(case["batch"], RUN["Ra_s"]))
        s["out"] = torch.empty_like(s["X"])
    elif kind == "newton":
        X, Ra = _newton_inputs(case, seed)
        s["plan"] = _plan(case, THIN["dt"], THIN, symmetric=True)
        s["krylov"] = newton.Krylov(s["plan"], restart=case["restart"])
        s["X"], s["Ra"], s["Ra_s"] = _dev(X[0]), _dev(Ra), _dev(np.array([THIN["Ra_s"]]))
    elif kind == "newtons":
        X, Ra = _newton_inputs(case, seed)
        s["plan"] = _plan(case, THIN["dt"], THIN, case["batch"], symmetric=True)
        s["solver"] = newton.NewtonBatch(s["plan"], restart=case["restart"],
                                         max_batch=case["batch"])
        s["X"], s["Ra"] = _dev(X), _dev(Ra)
        s["Ra_s"] = _dev(np.full(case["batch"], THIN["Ra_s"]))
    elif kind == "time_loop":
        s["X"], s["Ra"] = _time_loop_inputs(case, seed)
        s["file"] = os.path.join(tempfile.gettempdir(), "time_loop_%d.h5" % os.getpid())
    else:
        a, x = _transform_inputs(case, seed)
        s["a"], s["x"] = _dev(a), _dev(x)
        K, M, rows = case["N_fm"], x.shape[1], case["rows"]
        s["outs"] = [torch.empty((rows, n), dtype=torch.float64, device="cuda")
                     for n in (M, M, K, K)]
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["plan"].step(s["X"], s["Ra"], s["Ra_s"], nsteps=s["nsteps"], out=s["out"])
        return [s["out"], s["plan"].diagnostics(s["out"])] if s["monitor"] else [s["out"]]
    if kind == "graph":
        s["graph"].launch()
        return [s["X"]]
    if kind == "sweep":
        s["graph"].launch()
        return [c.X for c in s["sweep"].classes.values()]
    if kind == "linearised":
        return [s["plan"].step_linearized(s["v"], s["X"], s["Ra"], s["Ra_s"], out=s["out"])]
    if kind == "newton":
        return [s["krylov"].newton(s["X"], s["Ra"], s["Ra_s"])[0]]
    if kind == "newtons":
        return [s["solver"].solve(s["X"], s["Ra"], s["Ra_s"])[0]]
    if kind == "time_loop":
        p = RUN
        return [Main._Time_Step(s["X"], s["Ra"], p["Ra_s"], p["Tau"], p["Pr"], p["d"], s["N_fm"],
                                s["N_r"], s["symmetric"], save_filename=s["file"],
                                Total_time=(s["nsteps"] + 0.5) * p["dt"], dt=p["dt"])]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    K, M, rows = s["N_fm"], s["x"].shape[1], s["rows"]
    jobs = ((_lib.SDDC_IDCT, s["a"], K, M), (_lib.SDDC_IDST, s["a"], K, M),
            (_lib.SDDC_DCT, s["x"], M, K), (_lib.SDDC_DST, s["x"], M, K))
    for (what, src, n_in, n_out), dst in zip(jobs, s["outs"]):
        _lib.check(_lib.lib().sddc_transform(what, ctypes.c_void_p(src.data_ptr()),
                                             ctypes.c_void_p(dst.data_ptr()), rows, n_in, n_out,
                                             stream))
    return s["outs"]


# --------------------------------------------------------------------- work
def _step_flops(K, nr):
    """One instance-step: six Chebyshev contractions, the four products of the
    three solves, eleven length-M transforms per radial row."""
    M = 1.5 * K
    return (6 + 4) * 2.0 * K * nr * nr + 11 * nr * 2.5 * M * math.log2(M)


def _operator_bytes(K, nr):
    return 8.0 * (3 * K * nr * nr + 5 * nr * nr)


def work(case):
    kind = case["kind"]
    if kind == "transforms":
        K, rows = case["N_fm"], case["rows"]
        M = 3 * K // 2
        return {"bytes": 8.0 * rows * 3 * (K + M),
                "flops": 4 * rows * 2.5 * M * math.log2(M)}
    if kind == "sweep":
        # mean over the twelve classes
        sizes = [(K, r - 1) for r in (20, 30, 40) for K in (64, 128, 256, 512)]
        n = case["instances"] / len(sizes)
        return {"bytes": sum(n * 48.0 * K * nr + _operator_bytes(K, nr) for K, nr in sizes),
                "flops": case["nsteps"] * sum(n * _step_flops(K, nr) for K, nr in sizes)}
    K, nr, B = case["N_fm"], case["N_r"] - 1, case.get("batch", 1)
    state = 8.0 * 3 * K * nr
    if kind in ("step", "graph", "time_loop"):
        return {"bytes": 2 * B * state + _operator_bytes(K, nr),
                "flops": B * case["nsteps"] * _step_flops(K, nr)}
    if kind == "linearised":
        return {"bytes": 3 * B * state + _operator_bytes(K, nr), "flops": 2.0 * B * _step_flops(K, nr)}
    # two Newton iterations of about twenty J v each
    return {"bytes": 2 * B * state + _operator_bytes(K, nr), "flops": 80.0 * B * _step_flops(K, nr)}


# -------------------------------------------------------- the method in NumPy
class _Model:
    """Operators and step of one size class, states as arrays (B, 3, K, nr)."""

    def __init__(self, K, Nr, d, dt, Pr, Tau, symmetric=False):
        self.K, self.Nr, self.nr, self.d, self.dt, self.Pr, self.Tau = K, Nr, Nr - 1, d, dt, Pr, Tau
        self.symmetric = symmetric
        n = np.arange(Nr + 1)
        R1, R2 = 1.0 / d, (1.0 + d) / d
        R = 0.5 * (R1 + R2) + 0.5 * (R1 - R2) * np.cos(np.pi * n / Nr)
        c = np.where((n == 0) | (n == Nr), 2.0, 1.0) * (-1.0) ** n
        D = np.outer(c, 1.0 / c) / (R[:, None] - R[None, :] + np.eye(Nr + 1))
        D -= np.diag(D.sum(axis=1))
        self.D, self.R = D, R
        inner = slice(1, -1)
        r = R[inner]
        DD = D @ D
        self.Dr, self.D2s = D[inner, inner], DD[inner, inner]
        self.r, self.A_T = r, R1 * R2 / (R1 - R2)
        lap = (R[:, None] ** 2 * DD + 2.0 * R[:, None] * D)[inner, inner]
        # clamped fourth derivative: psi = q v with q = (r - R_1)(r - R_2)
        q = (R - R[0]) * (R - R[-1])
        s = np.zeros(Nr + 1)
        s[inner] = 1.0 / q[inner]
        D3, D4 = D @ DD, DD @ DD
        four = (q[:, None] * D4 + 4.0 * (2.0 * R - R[0] - R[-1])[:, None] * D3 + 12.0 * DD) * s
        four = four[inner, inner]
        D2 = ((2.0 * DD - 4.0 * D / R[:, None] + np.diag(6.0 / R ** 2)) / (R ** 2)[:, None])
        self.D2 = D2[inner, inner]
        j = np.arange(1, K + 1, dtype=np.float64)           # psi row k: sin (k+1) theta
        bj = (-j * (j + 1))[:, None, None]
        h = Pr * dt
        i2, i4 = np.diag(r ** -2.0), np.diag(r ** -4.0)
        self.inv_psi = np.linalg.inv(self.D2s + bj * i2 - h * (four + bj * (self.D2 + bj * i4)))
        k = np.arange(K, dtype=np.float64)                  # T, S row k: cos k theta
        bk = (-k * (k + 1))[:, None, None]
        eye = np.eye(Nr - 1)
        self.inv = [np.linalg.inv(np.diag(r ** 2) - t * (lap + bk * eye)) for t in (dt, Tau * dt)]
        M = 3 * K // 2
        th = np.pi * (2 * np.arange(M) + 1) / (2 * M)
        self.cos, self.sin = np.cos(np.outer(k, th)), np.sin(np.outer(k, th))
        self.M = M

    def mask(self, X):
        if not self.symmetric:
            return X
        X = X.copy()
        X[:, 0, 0::2] = 0.0
        X[:, 1:, 1::2] = 0.0
        return X

    def theta(self, psi):
        """J_theta psi, A2 psi and omega = A2 / r^2-type operator of psi."""
        K, r = self.K, self.r
        P = np.zeros_like(psi)
        for k in range(K - 3, -1, -1):
            P[:, k] = P[:, k + 2] + psi[:, k + 2]
        j = np.arange(1.0, K + 1)[:, None]
        t = (j + 1) * psi + 2 * P
        D2psi = psi @ self.D2s.T
        A2 = D2psi - j * t / r ** 2
        om = D2psi / r ** 2 - j * t / r ** 4
        Q = np.zeros_like(psi)
        Q[:, :-1] = psi[:, 1:] + P[:, 1:]
        J = 2 * Q
        J[:, 0] = Q[:, 0]
        J[:, 1:] += np.arange(2.0, K + 1)[:, None] * psi[:, :-1]
        return J, A2, om

    def _sine(self, a):
        """Rows k (sin (k+1) theta) to the sinusoid index, sin K theta dropped."""
        out = np.zeros_like(a)
        out[:, 1:] = a[:, :-1]
        return out

    def products(self, X):
        """F(X, X) as (B, 3, K, nr)."""
        K = self.K
        psi, T, S = X[:, 0], X[:, 1], X[:, 2]
        m = np.arange(K, dtype=np.float64)[:, None]
        J, _, om = self.theta(psi)
        om, Dp = self._sine(om), self._sine(psi @ self.Dr.T)
        C = lambda a: np.swapaxes(a, 1, 2) @ self.cos   # noqa: E731  (B, nr, M)
        Z = lambda a: np.swapaxes(a, 1, 2) @ self.sin   # noqa: E731
        gJ, gom, gDp = C(J), Z(om), Z(Dp)
        q = gJ * gom
        rr = C(m * Dp) * gom + gDp * C(m * om)
        nt = gJ * C(T @ self.Dr.T) - gDp * Z(-m * T)
        ns = gJ * C(S @ self.Dr.T) - gDp * Z(-m * S)
        a = 2.0 / self.M
        sine = lambda x: a * np.swapaxes(x @ self.sin.T, 1, 2)   # noqa: E731

        def cosine(x):
            y = a * np.swapaxes(x @ self.cos.T, 1, 2)
            y[:, 0] *= 0.5
            return y

        F = np.zeros_like(X)
        F[:, 0, :-1] = (sine(q) @ self.Dr.T - sine(rr))[:, 1:]
        F[:, 1], F[:, 2] = cosine(nt), cosine(ns)
        return F

    def solve_heat(self, g, inv, h):
        f = np.zeros_like(g)
        for s in (self.K - 1, self.K - 2):
            if self.symmetric and s % 2 == 1:
                continue
            b = np.zeros_like(g[:, 0])
            for j in range(s, -1, -2):
                f[:, j] = (g[:, j] - (0.5 if j == 0 else 1.0) * b) @ inv[j].T
                b = b + 2.0 * h * j * f[:, j]
        return f

    def solve_psi(self, g):
        f = np.zeros_like(g)
        h, i2, i4 = self.Pr * self.dt, self.r ** -2.0, self.r ** -4.0
        for s in (self.K - 1, self.K - 2):
            if self.symmetric and s % 2 == 0:
                continue
            fe = np.zeros_like(g[:, 0])
            le = np.zeros_like(fe)
            for row in range(s, -1, -2):
                j = row + 1.0
                bj, bt = -j * (j + 1), -2.0 * j
                b = h * bt * (fe @ self.D2.T + bj * i4 * fe + i4 * le) - bt * i2 * fe
                f[:, row] = (g[:, row] + b) @ self.inv_psi[row].T
                le = le + bj * f[:, row] + bt * fe
                fe = fe + f[:, row]
        return f

    def step(self, X, Ra, Ra_s):
        X = self.mask(X)
        psi, T, S = X[:, 0], X[:, 1], X[:, 2]
        J, A2, _ = self.theta(psi)
        r, dt = self.r, self.dt
        G = -dt * self.products(X)
        R1 = 1.0 / self.d
        G[:, 0] += A2
        j = np.arange(1.0, self.K)[:, None]
        buoy = Ra[:, None, None] * T[:, 1:] - Ra_s[:, None, None] * S[:, 1:]
        G[:, 0, :-1] += dt * self.Pr * (-j * R1 ** 2 / r ** 2) * buoy
        adv = dt * (self.A_T / r ** 2) * J
        G[:, 1] += r ** 2 * T - adv
        G[:, 2] += r ** 2 * S - adv
        return np.stack([self.solve_psi(G[:, 0]),
                         self.solve_heat(G[:, 1], self.inv[0], dt),
                         self.solve_heat(G[:, 2], self.inv[1], self.Tau * dt)], axis=1)

    def linearised(self, v, X, Ra, Ra_s):
        """The step is quadratic in X: its central difference is its derivative."""
        scale = np.sqrt((X ** 2).sum(axis=(1, 2, 3), keepdims=True)
                        / np.maximum((v ** 2).sum(axis=(1, 2, 3), keepdims=True), 1e-300))
        w = scale * v
        return (self.step(X + w, Ra, Ra_s) - self.step(X - w, Ra, Ra_s)) / (2.0 * scale)

    def diagnostics(self, X):
        K, nr, r, R = self.K, self.nr, self.r, self.R
        psi = X[:, 0]
        J, _, _ = self.theta(psi)
        L = 3 * K
        th = np.pi * (2 * np.arange(L) + 1) / (2 * L)
        k = np.arange(K)
        gJ = np.swapaxes(J / r, 1, 2) @ np.cos(np.outer(k, th))
        gD = np.swapaxes(self._sine(psi @ self.Dr.T), 1, 2) @ np.sin(np.outer(k, th))
        w = np.full(L, np.pi / L)
        w[[0, -1]] *= 0.5
        row = (gJ ** 2 + gD ** 2) @ (w * np.sin(th))
        V = (2.0 / 3.0) * (R[-1] ** 3 - R[0] ** 3)
        ke = (0.5 / V) * (0.5 * (row[:, 1:] + row[:, :-1]) * np.diff(r)).sum(axis=1)
        even = np.arange(0, K, 2)
        den = 1.0 - even.astype(np.float64) ** 2
        out = [np.sqrt((X ** 2).sum(axis=(1, 2, 3))), ke]
        for end in (0, -1):
            for f in (1, 2):
                flux = X[:, f, even] @ self.D[end, 1:-1]
                out.append(R[end] ** 2 / self.A_T * (flux / den).sum(axis=1))
        return np.stack(out, axis=1)

    def newton(self, X, Ra, Ra_s):
        """The steady state near X (B = 1) to rounding: Newton with GMRES."""
        X = self.mask(X)
        for _ in range(6):
            F = self.step(X, Ra, Ra_s) - X
            if np.linalg.norm(F) < 1e-14 * np.linalg.norm(X):
                break
            dv = self._gmres(lambda v: self.linearised(v, X, Ra, Ra_s) - v, F)
            X = X - dv
            if np.linalg.norm(dv) < 1e-11 * np.linalg.norm(X):
                break
        return X

    @staticmethod
    def _gmres(A, b, m=160, tol=1e-9):
        beta = np.linalg.norm(b)
        V = [b / beta]
        H = np.zeros((m + 1, m))
        for j in range(m):
            w = A(V[j])
            for _ in range(2):
                for i in range(j + 1):
                    h = float((V[i] * w).sum())
                    H[i, j] += h
                    w = w - h * V[i]
            H[j + 1, j] = np.linalg.norm(w)
            V.append(w / H[j + 1, j])
            e = np.zeros(j + 2)
            e[0] = beta
            y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)
            if np.linalg.norm(H[:j + 2, :j + 1] @ y - e) < tol * beta:
                break
        return sum(c * v for c, v in zip(y, V))


def _march(case, X, Ra, Ra_s, nsteps, symmetric):
    K, Nr = case["N_fm"], case["N_r"]
    m = _Model(K, Nr, RUN["d"], RUN["dt"], RUN["Pr"], RUN["Tau"], symmetric)
    X = X.reshape(X.shape[0], 3, K, Nr - 1)
    for _ in range(nsteps):
        X = m.step(X, Ra, Ra_s)
    return X, m


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "graph", "time_loop"):
        B = case.get("batch", 1)
        if B * case["nsteps"] * case["N_fm"] ** 2 * case["N_r"] > 3e9:
            return None   # over about 20 s in NumPy
        if kind == "time_loop":
            s = _time_loop_inputs(case, seed)
            X, Ra, nsteps = s[0][None], np.array([s[1]]), case["nsteps"]
        else:
            X, Ra = _run_inputs(case, seed)
            nsteps = case["nsteps"]
        X, m = _march(case, X, Ra, np.full(B, RUN["Ra_s"]), nsteps, case["symmetric"])
        flat = X.reshape(B, -1)
        if kind == "time_loop":
            return [flat[0]]
        return [flat, m.diagnostics(X)] if case.get("monitor") else [flat]
    if kind == "sweep":
        if case["instances"] * case["nsteps"] > 1300:
            return None
        groups = {}
        for inst in _sweep_inputs(case, seed):
            groups.setdefault((inst["N_fm"], inst["N_r"]), []).append(inst)
        outs = []
        for (K, Nr), g in groups.items():
            X, _ = _march(dict(N_fm=K, N_r=Nr), np.stack([i["X0"] for i in g]),
                          np.array([i["Ra"] for i in g]), np.array([i["Ra_s"] for i in g]),
                          case["nsteps"], False)
            outs.append(X.reshape(len(g), -1))
        return outs
    if kind == "linearised":
        X, v, Ra = _linearised_inputs(case, seed)
        K, nr, B = case["N_fm"], case["N_r"] - 1, case["batch"]
        m = _Model(K, case["N_r"], RUN["d"], 1.0, RUN["Pr"], RUN["Tau"], case["symmetric"])
        shape = (B, 3, K, nr)
        out = m.linearised(m.mask(v.reshape(shape)), m.mask(X.reshape(shape)), Ra,
                           np.full(B, RUN["Ra_s"]))
        return [out.reshape(B, -1)]
    if kind in ("newton", "newtons"):
        X, Ra = _newton_inputs(case, seed)
        K, nr, B = case["N_fm"], case["N_r"] - 1, X.shape[0]
        if B * K > 800:
            return None
        m = _Model(K, case["N_r"], THIN["d"], THIN["dt"], THIN["Pr"], THIN["Tau"], True)
        out = [m.newton(X[b].reshape(1, 3, K, nr), Ra[b:b + 1], np.array([THIN["Ra_s"]]))
               for b in range(B)]
        out = np.concatenate(out).reshape(B, -1)
        return [out[0] if kind == "newton" else out]
    a, x = _transform_inputs(case, seed)
    K, M = a.shape[1], x.shape[1]
    th = np.pi * (2 * np.arange(M) + 1) / (2 * M)
    k = np.arange(K)
    C, S = np.cos(np.outer(k, th)), np.sin(np.outer(k, th))
    dct = (2.0 / M) * x @ C.T
    dct[:, 0] *= 0.5
    return [a @ C, a @ S, dct, (2.0 / M) * x @ S.T]
