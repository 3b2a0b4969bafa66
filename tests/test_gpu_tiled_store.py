"""Tiled row stores (one-lane kernels, 4,096 instances and more) against the oracle and
against small batches, whose rows lie instance by instance, bit for bit: batches
around a tile of 64 slots, step caps around a block of four rows, rows of four to
seven doubles, a caller's system, the observed full store, and two seeds per sweep on
more lanes than a wave per SIMD."""
import ctypes as C
import dataclasses
import os

import numpy as np
import pytest

from helpers import run_oracle

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _same(a, b, what):
    a, b = np.asarray(a), np.asarray(b)
    assert np.array_equal(a, b, equal_nan=a.dtype == np.float64), what


def _against_oracle(out, o):
    import torch
    torch.cuda.synchronize()
    for k in ("status", "n_acc", "n_rej", "yT", "J", "dJdy0", "dJdp"):
        g, e = out[k].cpu().numpy(), o[k]
        if k in ("yT", "J"):  # what a failed forward leaves is not compared
            g, e = g[..., o["status"] == 0], e[..., o["status"] == 0]
        _same(g, e, k)


@pytest.mark.parametrize("B,max_steps", [(4096, 256), (4097, 257), (4159, 258), (4161, 259)])
def test_rows_match_oracle_in_either_order(B, max_steps):
    import oracle as O
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    w = dataclasses.replace(I.WORKLOADS["vdp"], t1=2.0)
    inp = I.make_inputs(w, B)
    pb = O.problem(w.system, w.n, w.np, w.tableau, t0=w.t0, t1=w.t1, dt0=w.dt0, abs_tol=w.tol,
                   rel_tol=w.tol, max_steps=max_steps)
    print(f"[gpu] tiled rows B={B} max_steps={max_steps}", flush=True)
    y0, p = _dev(inp["y0"]), _dev(inp["p"])
    with va.Solver(va.Problem.from_workload(w, batch=B, max_steps=max_steps)) as s:
        for _ in range(2):  # slot b is instance b's, then the k-th taken is in slot k
            s.forward(y0.clone(), p)
            for b in (0, 63, 64, B // 2, B - 65, B - 1):
                o = O.Solve(pb, inp["y0"][:, b].copy(), inp["p"][:, b].copy())
                rows = s.trajectory(b)
                _same(rows[:, 0], o.times, b)
                _same(rows[:-1, 1], np.diff(o.times), b)
                _same(rows[:, 2:], o.states, b)


@pytest.mark.parametrize("n", [2, 3, 4, 5])
@pytest.mark.parametrize("tableau", ["TAB_CASH_KARP54", "TAB_FEHLBERG78"])
def test_one_lane_lotka_volterra(n, tableau):
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    B = 4161
    w = dataclasses.replace(I.WORKLOADS["glv10"], n=n, np=n + n * n, t1=5.0,
                            tableau=getattr(va, tableau))
    inp = I.make_inputs(w, B)
    kw = dict(max_steps=1023, max_attempts=500)
    o = run_oracle(w, inp, **kw)
    print(f"[gpu] one-lane Lotka-Volterra N={n} {tableau} B={B}", flush=True)
    with va.Solver(va.Problem.from_workload(w, batch=B, instances_per_wave=64, **kw)) as s:
        for _ in range(2):
            _against_oracle(s.solve(_dev(inp["y0"]), _dev(inp["p"]), w.cost), o)


def test_callers_system():
    import oracle as O
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    lib = C.CDLL(os.path.join(ROOT, "tests", "cpp", "libva_user_system.so"))
    lib.va_brusselator_kernels.restype = C.c_void_p
    lib.va_brusselator_kernels.argtypes = [C.c_int32, C.c_int32]
    host = C.CDLL(os.path.join(ROOT, "tests", "cpp", "libva_brusselator_host.so"))
    O.set_user_system(host.brusselator_rhs, host.brusselator_vjp)
    B = 4161
    w = dataclasses.replace(I.WORKLOADS["brusselator"], t1=5.0)
    inp = I.make_inputs(w, B)
    o = run_oracle(w, inp, max_steps=1023)
    print(f"[gpu] caller's system, tiled, B={B}", flush=True)
    pb = va.Problem.from_workload(w, batch=B, max_steps=1023)
    with va.Solver(pb, kernels=lib.va_brusselator_kernels(w.tableau, 1)) as s:
        for _ in range(2):
            _against_oracle(s.solve(_dev(inp["y0"]), _dev(inp["p"]), w.cost), o)


# 66,001: more lanes than a wave per SIMD, compared through its first and last instances
@pytest.mark.parametrize("B", [4161, 66001])
def test_observed_full_store(B):
    import oracle as O
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    K, t1 = 7, 2.0
    w = dataclasses.replace(I.WORKLOADS["vdp_obs"], t1=t1)
    inp = I.make_inputs(w, B)
    inp["p"] = np.minimum(inp["p"], 20.0)
    few = np.r_[0:300, B - 300:B] if B > 10000 else np.arange(B)
    t_obs = t1 * np.arange(1, K + 1) / K
    y_obs = np.stack([2 * np.cos(t_obs), -2 * np.sin(t_obs)], axis=1)
    kw = dict(t1=t1, max_steps=1022)
    pb = O.problem(w.system, w.n, w.np, w.tableau, t0=w.t0, dt0=w.dt0, abs_tol=w.tol,
                   rel_tol=w.tol, **kw)
    o = O.solve_batch(pb, inp["y0"][:, few].copy(), inp["p"][:, few].copy(), 0,
                      obs=(t_obs, y_obs), nthreads=8)
    print(f"[gpu] observed full store B={B}", flush=True)
    with va.Solver(va.Problem.from_workload(w, batch=B, n_obs=K, **kw)) as s:
        for _ in range(2):
            out = s.solve_observed(_dev(inp["y0"]), _dev(inp["p"]), _dev(t_obs), _dev(y_obs))
            _against_oracle({k: v[..., few] for k, v in out.items()}, o)
            for b in (0, 64, B - 1):
                rows = s.trajectory(b)
                e = O.Solve(pb, inp["y0"][:, b].copy(), inp["p"][:, b].copy(),
                            obs=(t_obs, y_obs))
                _same(rows[:, 0], e.times, b)
                _same(rows[:, 2:], e.states, b)


# two seeds per sweep where the state has room for them, else in turn (N = 5)
@pytest.mark.parametrize("system,n,ipw", [("vdp", 2, 0), ("glv10", 2, 64), ("glv10", 5, 64)])
@pytest.mark.parametrize("nout", [2, 3])
def test_seeds_on_many_lanes(system, n, ipw, nout):
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    B = 66001
    w = dataclasses.replace(I.WORKLOADS[system], t1=0.5)
    if system == "glv10":
        w = dataclasses.replace(w, n=n, np=n + n * n)
    inp = I.make_inputs(w, B)
    few = np.r_[0:200, B - 200:B]
    rng = np.random.default_rng(3)
    lam0, mu0 = rng.normal(size=(nout, n, B)), rng.normal(size=(nout, w.np, B))
    print(f"[gpu] {nout} seeds {system} N={n} B={B}", flush=True)
    got = []
    for cols in (np.arange(B), few):
        y0, p = _dev(inp["y0"][:, cols]), _dev(inp["p"][:, cols])
        pb = va.Problem.from_workload(w, batch=cols.size, max_steps=255, instances_per_wave=ipw)
        with va.Solver(pb) as s:
            for _ in range(2):
                s.forward(y0.clone(), p)
            lam, mu = s.adjoint(p, _dev(lam0[..., cols]), _dev(mu0[..., cols]))
            S = s.sensitivity_matrix(p)
            torch.cuda.synchronize()
            got.append([t.cpu().numpy() for t in (lam, mu, S)])
    for a, b in zip(*got):
        _same(a[..., few], b, (system, nout))
