"""Performance cases: the solves that users of this library run, through its public
Python entry points (vectorizedadjoint_amd.Solver and odeint_adjoint).

listed() names the cases, draw(rng) gives more of the same ranges, prepare(case, seed)
builds a handle and its inputs on the GPU, run(state) makes one pass and returns every
output, work(case) counts the bytes and operations the pass cannot do without, and
exact(case, seed) is the same result in plain torch float64.
"""
from __future__ import annotations

import math

import torch

import vectorizedadjoint_amd as va
from vectorizedadjoint_amd import constants as K
from vectorizedadjoint_amd import flops as FL
from vectorizedadjoint_amd.autograd import odeint_adjoint

TABLEAUS = {"rk4": K.TAB_RK4, "cash_karp54": K.TAB_CASH_KARP54, "dopri5": K.TAB_DOPRI5,
            "fehlberg78": K.TAB_FEHLBERG78}
COSTS = {"sum": K.COST_SUM, "squared_norm": K.COST_SQUARED_NORM}

# "call" is what one pass runs:
#   solve       Solver.solve: forward, terminal cost, adjoint
#   adjoint     Solver.forward, then Solver.adjoint with one seed per state (the drop-in
#               runge_kutta / adjointSolve pair)
#   sensitivity Solver.forward, then Solver.sensitivity_matrix
#   autograd    odeint_adjoint under a loss, gradients by torch.autograd
#   observed    Solver.solve_observed
#   shared      Solver.solve_shared


def _vdp(name, B, **kw):
    c = dict(system="vdp", call="solve", n=2, batch=B, tableau="dopri5", tol=1e-8, t1=20.0,
             dt0=1e-3, mu_lo=0.5, mu_hi=5.0, cost="squared_norm", max_steps=2048, flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def _osc(name, B, **kw):
    c = dict(system="oscillator", call="solve", n=2, batch=B, tableau="dopri5", tol=1e-10,
             t1=30.0, dt0=1e-3, cost="squared_norm", max_steps=1536, flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def _osc_rk4(name, B, **kw):
    c = dict(system="oscillator_fixed_k", call="adjoint", n=2, batch=B, tableau="rk4", tol=0.0,
             t1=10.0, dt0=0.01, cost="sum", max_steps=1024, flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def _glv(name, B, n=10, **kw):
    c = dict(system="glv", call="solve", n=n, batch=B, tableau="cash_karp54", tol=1e-8, t1=50.0,
             dt0=1e-3, cost="sum", max_steps=1024, flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def _obs(name, B, **kw):
    c = dict(system="vdp", call="observed", n=2, batch=B, tableau="dopri5", tol=1e-8, t1=20.0,
             dt0=1e-3, mu_lo=0.1, mu_hi=100.0, n_obs=50, cost="sum", max_steps=8192, budget=0,
             flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def _shared(name, B, **kw):
    c = dict(system="glv_shared", call="shared", n=128, batch=B, tableau="cash_karp54", tol=1e-8,
             t1=50.0, dt0=1e-3, cost="sum", max_steps=512, flags=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One trajectory and its full Jacobian, as a caller of the one-instance Driver has it
        # (the Van der Pol example: mu = 1e3, Fehlberg 7(8), tol 1e-5): pure latency.
        _vdp("vdp_single", 1, call="adjoint", tableau="fehlberg78", tol=1e-5, t1=0.5,
             mu_lo=1000.0, mu_hi=1000.0),
        # A small ensemble, far from filling the chip: the chain of one instance's steps.
        _vdp("vdp_1k", 1024),
        # The largest ensemble: every lane busy, 25 GB of trajectory rows.
        _osc("oscillator_1m", 1 << 20),
        # Fixed steps without a controller (the harmonic oscillator example's RK4 run).
        _osc_rk4("oscillator_rk4_40k", 40000),
        # The headline workload: repeated solves of one parameter sweep on one handle.
        _glv("glv10_64k", 65536),
        # The same model over batches that have nothing to do with each other, in index order.
        _glv("glv10_unrelated_20k", 20011, flags=int(K.FLAG_COLD_ORDER)),
        # A fitting loop's step: forward and backward through torch.autograd.
        _glv("glv10_fit_4k", 4096, call="autograd", t1=10.0),
        # Sensitivity matrices: one seed per state component.
        _glv("glv5_sensitivity_8k", 8192, n=5, call="sensitivity", t1=10.0),
        # An odd number of species, another tableau, a ragged batch.
        _glv("glv13_dopri5_5k", 5003, n=13, tableau="dopri5", t1=10.0),
        # Calibration against observation times under a 4 GB trajectory budget (checkpointed).
        _obs("vdp_observed_256k", 262144, budget=4 << 30, max_steps=16384),
        # The same cost on a batch whose trajectories are stored in full.
        _obs("vdp_observed_6k", 6000, mu_hi=10.0, n_obs=20, max_steps=2048),
        # An interaction matrix shared by the whole batch (FP64 matrix instructions).
        _shared("glv128_shared_16k", 16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vdp", "vdp", "oscillator", "oscillator", "rk4", "glv", "glv", "glv",
                       "fit", "sensitivity", "observed", "observed", "shared"])
    if kind == "vdp":
        tab = rng.choice(["dopri5", "cash_karp54", "fehlberg78"])
        return _vdp(None, _log_int(rng, 1, 200000), tableau=tab, tol=10.0 ** -rng.uniform(6, 9),
                    t1=rng.uniform(5.0, 20.0), call=rng.choice(["solve", "solve", "adjoint"]),
                    flags=int(rng.choice([0, 0, K.FLAG_GRAPH])))
    if kind == "oscillator":
        return _osc(None, _log_int(rng, 100, 1 << 20),
                    tableau=rng.choice(["dopri5", "dopri5", "cash_karp54", "fehlberg78"]),
                    tol=10.0 ** -rng.uniform(6, 10), t1=rng.uniform(10.0, 30.0))
    if kind == "rk4":
        return _osc_rk4(None, _log_int(rng, 64, 200000), t1=rng.uniform(2.0, 10.0))
    if kind in ("glv", "fit", "sensitivity"):
        n = rng.randint(2, 24) if kind == "glv" else rng.choice([3, 4, 5, 7, 10])
        top = {"glv": 65536, "fit": 16384, "sensitivity": 16384}[kind] * min(1.0, (10.0 / n) ** 2)
        call = {"glv": "solve", "fit": "autograd", "sensitivity": "sensitivity"}[kind]
        return _glv(None, _log_int(rng, 16, max(64, int(top))), n=n, call=call,
                    tableau=rng.choice(["cash_karp54", "cash_karp54", "dopri5", "fehlberg78"]),
                    tol=10.0 ** -rng.uniform(6, 9), t1=rng.uniform(5.0, 15.0),
                    flags=int(rng.choice([0, 0, K.FLAG_COLD_ORDER])))
    if kind == "observed":
        B = _log_int(rng, 64, 262144)
        full = B <= 16384 and rng.random() < 0.5
        return _obs(None, B, mu_hi=10.0 if full else rng.choice([10.0, 100.0]),
                    n_obs=rng.randint(5, 60), max_steps=4096 if full else 16384,
                    budget=0 if full else max(1 << 28, B * (4 << 30) // 262144))
    return _shared(None, _log_int(rng, 16, 16384), t1=rng.uniform(10.0, 50.0),
                   tableau=rng.choice(["cash_karp54", "cash_karp54", "dopri5"]))


# ---------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _normal(g, s, *shape):
    return s * torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _inputs(case, seed):
    """y0 [N, B], p [P, B] (for the shared model r [N, B], and A [N, N]) with the
    distributions of vectorizedadjoint_amd.inputs."""
    g, B, n = _gen(seed), case["batch"], case["n"]
    if case["system"] == "vdp":
        lo, hi = case["mu_lo"], case["mu_hi"]
        if case["call"] == "observed":  # mu log-uniform: step counts over two decades
            p = torch.exp(_uniform(g, math.log(lo), math.log(hi), 1, B))
        else:
            p = _uniform(g, lo, hi, 1, B)
        y0 = _normal(g, 0.01, 2, B)
        y0[0] += 2.0
        return y0, p, None
    if case["system"] == "oscillator":
        p = torch.cat([_uniform(g, 0.5, 4.0, 1, B), _uniform(g, 0.0, 0.5, 1, B)])
        return _uniform(g, -1.0, 1.0, 2, B), p, None
    if case["system"] == "oscillator_fixed_k":
        return _uniform(g, -1.0, 1.0, 2, B), _uniform(g, 0.0, 0.5, 1, B), None
    if case["system"] == "glv":
        r = _uniform(g, 0.1, 1.0, n, B)
        # interactions scaled so that a larger community stays as stable as ten species
        A = _normal(g, 0.2 * math.sqrt(10.0 / max(10, n)), n, n, B)
        i = torch.arange(n, device="cuda")
        A[i, i] = -_uniform(g, 0.5, 1.5, n, B)
        return _uniform(g, 0.1, 1.0, n, B), torch.cat([r, A.reshape(n * n, B)]), None
    A = _normal(g, 0.05, n, n)
    A.fill_diagonal_(-1.0)
    return _uniform(g, 0.05, 0.5, n, B), _uniform(g, 0.1, 1.0, n, B), A


def _observations(case):
    k = case["n_obs"]
    t = case["t1"] * torch.arange(1, k + 1, dtype=torch.float64, device="cuda") / k
    return t, torch.stack([2.0 * torch.cos(t), -2.0 * torch.sin(t)], dim=1).contiguous()


SYSTEMS = {"vdp": K.SYS_VAN_DER_POL, "oscillator": K.SYS_OSCILLATOR,
           "oscillator_fixed_k": K.SYS_OSCILLATOR_FIXED_K, "glv": K.SYS_LOTKA_VOLTERRA,
           "glv_shared": K.SYS_LOTKA_VOLTERRA_SHARED}
FIXED_K = 1.0


def _n_param(case):
    n = case["n"]
    return {"vdp": 1, "oscillator": 2, "oscillator_fixed_k": 1, "glv": n + n * n,
            "glv_shared": n}[case["system"]]


def prepare(case, seed):
    y0, p, A = _inputs(case, seed)
    pb = va.Problem(system=SYSTEMS[case["system"]], n_state=case["n"], n_param=_n_param(case),
                    tableau=TABLEAUS[case["tableau"]], batch=case["batch"], t0=0.0,
                    t1=case["t1"], dt0=case["dt0"], abs_tol=case["tol"], rel_tol=case["tol"],
                    adaptive=case["tableau"] != "rk4", system_constant=FIXED_K,
                    max_steps=case["max_steps"], n_obs=case.get("n_obs", 0),
                    trajectory_budget_bytes=case.get("budget", 0), flags=case["flags"])
    st = {"case": case, "solver": va.Solver(pb), "y0": y0.contiguous(), "p": p.contiguous(),
          "A": A, "out": None, "cost": COSTS[case["cost"]]}
    n, P, B = case["n"], _n_param(case), case["batch"]
    if case["call"] == "observed":
        st["obs"] = _observations(case)
    elif case["call"] == "adjoint":
        st["seeds"] = torch.eye(n, dtype=torch.float64, device="cuda")[:, :, None].expand(
            n, n, B).contiguous()
        st["y"], st["lam"] = torch.empty_like(st["y0"]), torch.empty_like(st["seeds"])
        st["mu"] = torch.empty((n, P, B), dtype=torch.float64, device="cuda")
    elif case["call"] == "sensitivity":
        st["y"] = torch.empty_like(st["y0"])
    elif case["call"] == "autograd":
        st["y0"].requires_grad_()
        st["p"].requires_grad_()
        st["target"] = torch.full_like(y0, 0.5)
    return st


def run(st):
    s, call = st["solver"], st["case"]["call"]
    if call == "solve":
        st["out"] = s.solve(st["y0"], st["p"], st["cost"], out=st["out"])
        return st["out"]
    if call == "observed":
        st["out"] = s.solve_observed(st["y0"], st["p"], *st["obs"], out=st["out"])
        return st["out"]
    if call == "shared":
        st["out"] = s.solve_shared(st["y0"], st["p"], st["A"], st["cost"], out=st["out"])
        return st["out"]
    if call == "autograd":
        yT = odeint_adjoint(s, st["y0"], st["p"])
        loss = ((yT - st["target"]) ** 2).mean()
        gy, gp = torch.autograd.grad(loss, (st["y0"], st["p"]))
        return {"loss": loss.detach(), "yT": yT.detach(), "dy0": gy, "dp": gp}
    y = s.forward(st["y"].copy_(st["y0"]), st["p"])
    if call == "sensitivity":
        return {"yT": y, "S": s.sensitivity_matrix(st["p"])}
    lam, mu = s.adjoint(st["p"], st["lam"].copy_(st["seeds"]), st["mu"].zero_())
    return {"yT": y, "lam": lam, "mu": mu}


# ---------------------------------------------------------------------------- work

# mean accepted steps per unit of time at tol 1e-8 and the order the tolerance enters with
RATES = {("vdp", "dopri5"): (37.5, 5), ("vdp", "cash_karp54"): (30.4, 5),
         ("vdp", "fehlberg78"): (10.0, 8), ("oscillator", "dopri5"): (10.0, 5),
         ("oscillator", "cash_karp54"): (8.2, 5), ("oscillator", "fehlberg78"): (2.3, 8),
         ("glv", "cash_karp54"): (3.5, 5), ("glv", "dopri5"): (4.3, 5),
         ("glv", "fehlberg78"): (1.6, 8), ("glv_shared", "cash_karp54"): (2.0, 5),
         ("glv_shared", "dopri5"): (2.5, 5)}


def _mean_steps(case):
    if case["tableau"] == "rk4":
        return case["t1"] / case["dt0"]
    rate, q = RATES[case["system"], case["tableau"]]
    t1 = case["t1"]
    if case["system"] == "glv":  # the transient takes most of the steps
        t1 = min(t1, 10.0 + 0.3 * (t1 - 10.0)) if t1 > 10.0 else t1
    s = rate * t1 * (1e-8 / case["tol"]) ** (1.0 / q)
    if case["system"] == "vdp":  # steps grow with mu; the rates are for mu in [0.5, 5]
        lo, hi = case["mu_lo"], case["mu_hi"]
        mean = (hi - lo) / math.log(hi / lo) if case["call"] == "observed" else 0.5 * (lo + hi)
        s *= 0.4 + 0.22 * mean
    return s


def work(case):
    n, P, B = case["n"], _n_param(case), case["batch"]
    steps = _mean_steps(case)
    sysid, tab = SYSTEMS[case["system"]], TABLEAUS[case["tableau"]]
    seeds = n if case["call"] in ("adjoint", "sensitivity") else 1
    fwd = steps * FL.per_attempt_forward(sysid, n, tab)
    rev = steps * FL.per_step_reverse(sysid, n, tab)
    # y0, p in; y(T), the gradients and the per-instance scalars out
    doubles = B * (2 * n + P + seeds * (n + P) + 2)
    if case["system"] == "glv_shared":
        doubles += 2 * n * n
    return {"bytes": 8.0 * doubles, "flops": float(B) * (fwd + seeds * rev)}


# ---------------------------------------------------------------------------- exact

def _coefficients(tab):
    F = float
    if tab == "rk4":
        a = [[], [F(1) / 2], [0, F(1) / 2], [0, 0, 1.0]]
        return a, [1 / 6, 1 / 3, 1 / 3, 1 / 6], None, 4, 0
    if tab == "cash_karp54":
        a = [[], [1 / 5], [3 / 40, 9 / 40], [3 / 10, -9 / 10, 6 / 5],
             [-11 / 54, 5 / 2, -70 / 27, 35 / 27],
             [1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096]]
        b = [37 / 378, 0, 250 / 621, 125 / 594, 0, 512 / 1771]
        e = [2825 / 27648, 0, 18575 / 48384, 13525 / 55296, 277 / 14336, 1 / 4]
        return a, b, [x - y for x, y in zip(b, e)], 5, 4
    if tab == "dopri5":
        a = [[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
             [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
             [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
             [35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
        b = [35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84, 0]
        e = [5179 / 57600, 0, 7571 / 16695, 393 / 640, -92097 / 339200, 187 / 2100, 1 / 40]
        return a, b, [x - y for x, y in zip(b, e)], 5, 4
    a = [[], [2 / 27], [1 / 36, 1 / 12], [1 / 24, 0, 1 / 8], [5 / 12, 0, -25 / 16, 25 / 16],
         [1 / 20, 0, 0, 1 / 4, 1 / 5], [-25 / 108, 0, 0, 125 / 108, -65 / 27, 125 / 54],
         [31 / 300, 0, 0, 0, 61 / 225, -2 / 9, 13 / 900],
         [2, 0, 0, -53 / 6, 704 / 45, -107 / 9, 67 / 90, 3],
         [-91 / 108, 0, 0, 23 / 108, -976 / 135, 311 / 54, -19 / 60, 17 / 6, -1 / 12],
         [2383 / 4100, 0, 0, -341 / 164, 4496 / 1025, -301 / 82, 2133 / 4100, 45 / 82, 45 / 164,
          18 / 41],
         [3 / 205, 0, 0, 0, 0, -6 / 41, -3 / 205, -3 / 41, 3 / 41, 6 / 41, 0],
         [-1777 / 4100, 0, 0, -341 / 164, 4496 / 1025, -289 / 82, 2193 / 4100, 51 / 82, 33 / 164,
          12 / 41, 0, 1]]
    b = [0, 0, 0, 0, 0, 34 / 105, 9 / 35, 9 / 35, 9 / 280, 9 / 280, 0, 41 / 840, 41 / 840]
    db = [0.0] * 13
    db[0], db[10], db[11], db[12] = -41 / 840, -41 / 840, 41 / 840, 41 / 840
    return a, b, db, 8, 7


def _model(case, p, A):
    """rhs(x, idx) and vjp(x, w, idx) -> (w df/dx, w df/dp) over the instances idx."""
    n, kind = case["n"], case["system"]
    if kind == "vdp":
        def rhs(x, i):
            return torch.stack([x[1], p[0, i] * ((1 - x[0] ** 2) * x[1] - x[0])])

        def vjp(x, w, i):
            q = 1 - x[0] ** 2
            wm = w[1] * p[0, i]
            return (torch.stack([wm * (-2 * x[0] * x[1] - 1), wm * q + w[0]]),
                    (w[1] * (q * x[1] - x[0]))[None])
        return rhs, vjp
    if kind.startswith("oscillator"):
        both = kind == "oscillator"

        def kc(i):
            return (p[0, i], p[1, i]) if both else (FIXED_K, p[0, i])

        def rhs(x, i):
            k, c = kc(i)
            return torch.stack([x[1], -k * x[0] - c * x[1]])

        def vjp(x, w, i):
            k, c = kc(i)
            dc = -w[1] * x[1]
            return (torch.stack([-w[1] * k, w[0] - w[1] * c]),
                    torch.stack([-w[1] * x[0], dc]) if both else dc[None])
        return rhs, vjp
    if kind == "glv":
        def growth(x, i):
            q = p[:, i]
            return q, q[:n] + (q[n:].view(n, n, -1) * x[None]).sum(1)

        def rhs(x, i):
            return x * growth(x, i)[1]

        def vjp(x, w, i):
            q, g = growth(x, i)
            u = w * x
            wx = w * g + (q[n:].view(n, n, -1) * u[:, None]).sum(0)
            return wx, torch.cat([u, (u[:, None] * x[None]).reshape(n * n, -1)])
        return rhs, vjp

    def rhs_s(x, i):
        return x * (p[:, i] + A @ x)

    def vjp_s(x, w, i):
        u = w * x
        return w * (p[:, i] + A @ x) + A.t() @ u, u
    return rhs_s, vjp_s


def _forward64(case, rhs, y0):
    """The controlled (or fixed-step) loop, all instances an attempt at a time.  Returns the
    stored points (t [T, B], y [T, N, B]), the accepted counts, which ended well, the final
    states and the stored index of every observation."""
    a, b, db, order, err_order = _coefficients(case["tableau"])
    n, B, cap, t1 = case["n"], case["batch"], case["max_steps"], case["t1"]
    dev, f64 = "cuda", torch.float64
    eps = 2.220446049250313e-16
    K_obs = case.get("n_obs", 0)
    t_obs = _observations(case)[0] if K_obs else torch.empty(0, dtype=f64, device=dev)
    targets = torch.cat([t_obs, torch.tensor([t1], dtype=f64, device=dev)])
    rows = cap + 1 if db is not None else int(round(t1 / case["dt0"])) + 2
    T = torch.empty((rows, B), dtype=f64, device=dev)
    Y = torch.empty((rows, n, B), dtype=f64, device=dev)
    yT = torch.empty_like(y0)
    n_acc = torch.zeros(B, dtype=torch.long, device=dev)
    ok = torch.zeros(B, dtype=torch.bool, device=dev)
    points = torch.full((max(K_obs, 1), B), -1, dtype=torch.long, device=dev)

    def attempt(y, h, i):
        ks = []
        for row in a:
            x = y
            for c, k in zip(row, ks):
                if c:
                    x = x + (c * h) * k
            ks.append(rhs(x, i))
        new = y
        for c, k in zip(b, ks):
            if c:
                new = new + (c * h) * k
        return ks, new

    if db is None:
        i = torch.arange(B, device=dev)
        y, h, count = y0, case["dt0"], 0
        t = 0.0
        T[0], Y[0] = 0.0, y
        while t + h - t1 <= eps:
            _, y = attempt(y, torch.full((B,), h, dtype=f64, device=dev), i)
            count += 1
            t = count * h
            T[count], Y[count] = t, y
        n_acc[:] = count
        ok[:] = True
        return T, Y, n_acc, ok, y, points
    i = torch.arange(B, device=dev)
    y, t = y0.clone(), torch.zeros(B, dtype=f64, device=dev)
    h = torch.full((B,), case["dt0"], dtype=f64, device=dev)
    keep, clipped = h.clone(), torch.zeros(B, dtype=torch.bool, device=dev)
    fresh = torch.ones(B, dtype=torch.bool, device=dev)
    count, kobs = n_acc.clone(), n_acc.clone()
    trip = 0
    while i.numel():
        if K_obs:
            at = fresh & (kobs < K_obs) & ~(targets[kobs] - t > eps)
            while bool(at.any()):
                points[kobs[at], i[at]] = count[at]
                kobs = kobs + at
                at = at & (kobs < K_obs) & ~(targets[kobs] - t > eps)
        target = targets[kobs]
        done = fresh & ~(target - t > eps)
        over = fresh & ~done & (count >= cap)
        put = fresh & ~over
        T[count[put], i[put]] = t[put]
        Y[count[put], :, i[put]] = y[:, put].t()
        if trip % 8 == 0 or K_obs:
            stop = done | over
            if bool(stop.any()):
                j = i[stop]
                yT[:, j], n_acc[j] = y[:, stop], count[stop]
                ok[j] = done[stop] & torch.isfinite(y[:, stop]).all(0)
                go = ~stop
                i, y, t, h, keep = i[go], y[:, go], t[go], h[go], keep[go]
                clipped, fresh, count, kobs = clipped[go], fresh[go], count[go], kobs[go]
                target, done, over = target[go], done[go], over[go]
                if not i.numel():
                    break
        trip += 1
        clip = fresh & (t + h - target > eps)
        keep = torch.where(fresh, h, keep)
        clipped = torch.where(fresh, clip & (kobs < K_obs), clipped)
        h = torch.where(clip, target - t, h)
        ks, new = attempt(y, h, i)
        xe = sum((c * h) * k for c, k in zip(db, ks) if c)
        ratio = xe.abs() / (case["tol"] + case["tol"] * (y.abs() + h * ks[0].abs()))
        err = torch.nan_to_num(ratio, nan=0.0, posinf=math.inf).amax(0)
        good = ~(err > 1.0)
        grow = 0.9 * torch.clamp(err, min=5.0 ** -order) ** (-1.0 / order)
        cut = torch.clamp(0.9 * err ** (-1.0 / (err_order - 1)), min=0.2)
        h_next = torch.where(good, torch.where(err < 0.5, h * grow, h), h * cut)
        h_next = torch.where(good & clipped, torch.maximum(h_next, keep), h_next)
        clipped = clipped & good
        idle = done | over  # ended, not yet taken out
        step = good & ~idle
        t = torch.where(step, t + h, t)
        y = torch.where(step, new, y)
        h = torch.where(idle, h, h_next)
        count = count + step
        fresh = step | idle
    return T, Y, n_acc, ok, yT, points


def _reverse64(case, rhs, vjp, T, Y, n_acc, ok, points, lam, obs_y=None):
    """Discrete adjoint of the stored steps; lam [N, B] seeds.  Returns dJ/dy0, dJ/dp and, for
    the shared model, the summed dJ/dA."""
    a, b, _, _, _ = _coefficients(case["tableau"])
    n, B = case["n"], case["batch"]
    S = 6 if case["tableau"] == "dopri5" else len(a)
    mu = torch.zeros((_n_param(case), B), dtype=torch.float64, device="cuda")
    dA = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    lam = lam.clone()
    longest = torch.where(ok, n_acc, torch.full_like(n_acc, -1))
    order = torch.argsort(longest, descending=True)
    sorted_len = longest[order].cpu()
    live = 0
    if obs_y is not None:
        kobs = torch.full((B,), case["n_obs"] - 1, dtype=torch.long, device="cuda")

        def jumps(k):
            while True:
                c = kobs.clamp(min=0)
                hit = (kobs >= 0) & ok & (points.gather(0, c[None])[0] == k)
                j = hit.nonzero()[:, 0]
                if not j.numel():
                    return
                lam[:, j] += 2.0 * (Y[k, :, j] - obs_y[kobs[j]].t())
                kobs[j] -= 1
    for k in range(int(sorted_len[0]) if B else -1, -1, -1):
        if obs_y is not None:
            jumps(k + 1)
        while live < B and int(sorted_len[live]) > k:
            live += 1
        if not live:
            continue
        i = order[:live]
        h, y, l = T[k + 1, i] - T[k, i], Y[k][:, i], lam[:, i]
        xs, ks = [], []
        for m in range(S):
            x = y
            for c, q in zip(a[m], ks):
                if c:
                    x = x + (c * h) * q
            xs.append(x)
            ks.append(rhs(x, i))
        kb = [(b[m] * h) * l for m in range(S)]
        yb, acc = l, 0.0
        for m in range(S - 1, -1, -1):
            wx, wp = vjp(xs[m], kb[m], i)
            yb, acc = yb + wx, acc + wp
            if case["system"] == "glv_shared":
                dA += (kb[m] * xs[m]) @ xs[m].t()
            for j, c in enumerate(a[m][:m]):
                if c:
                    kb[j] = kb[j] + (wx * c) * h
        lam[:, i] = yb
        mu[:, i] += acc
    if obs_y is not None:
        jumps(0)
    lam[:, ~ok], mu[:, ~ok] = math.nan, math.nan
    return lam, mu, dA


def exact(case, seed):
    # A stiff observed batch takes some 7,500 steps one after the other: over 20 seconds here.
    if case["call"] == "observed" and case["mu_hi"] > 10.0:
        return None
    if case["batch"] * (case["max_steps"] + 1) * (case["n"] + 1) * 8 > 60e9:
        return None
    with torch.no_grad():
        y0, p, A = _inputs(case, seed)
        rhs, vjp = _model(case, p, A)
        T, Y, n_acc, ok, yT, points = _forward64(case, rhs, y0)
        bad = torch.where(ok, 0.0, math.nan)

        def back(lam, obs_y=None):
            return _reverse64(case, rhs, vjp, T, Y, n_acc, ok, points, lam, obs_y)
        call, n = case["call"], case["n"]
        if call in ("adjoint", "sensitivity"):
            lams, mus = [], []
            for o in range(n):
                seed_o = torch.zeros_like(y0)
                seed_o[o] = 1.0
                lam, mu, _ = back(seed_o)
                lams.append(lam)
                mus.append(mu)
            if call == "sensitivity":
                return {"yT": yT, "S": torch.stack(mus)}
            return {"yT": yT, "lam": torch.stack(lams), "mu": torch.stack(mus)}
        if call == "autograd":
            d = yT - 0.5
            lam, mu, _ = back(2.0 * d / d.numel())
            return {"loss": (d ** 2).mean(), "yT": yT, "dy0": lam, "dp": mu}
        ints = {"n_acc": None, "n_rej": None, "status": None}
        if call == "observed":
            obs_y = _observations(case)[1]
            J = torch.zeros_like(yT[0])
            for k in range(case["n_obs"]):
                at = points[k].clamp(min=0)
                yk = torch.stack([Y[:, c].gather(0, at[None])[0] for c in range(n)])
                J = J + ((yk - obs_y[k][:, None]) ** 2).sum(0)
            lam, mu, _ = back(torch.zeros_like(yT), obs_y)
            return dict(ints, J=J + bad, yT=yT, dJdy0=lam, dJdp=mu)
        if case["cost"] == "sum":
            J, lam = yT.sum(0), torch.ones_like(yT)
        else:
            J, lam = (yT ** 2).sum(0), 2.0 * yT
        lam, mu, dA = back(lam)
        if call == "shared":
            return dict(ints, J=J + bad, yT=yT, dJdy0=lam, dJdr=mu, dJdA=dA)
        return dict(ints, J=J + bad, yT=yT, dJdy0=lam, dJdp=mu)
