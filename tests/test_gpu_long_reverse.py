"""Reverses of instances that run long, three waves of a block each: the first solve
of a handle (index order, the head of the reverse's order in blocks of their own) and
the second (the long instances beside the bulk) against the oracle, bit for bit.

The number of species decides how the waves hold an instance: up to 16 the adjoint's
broadcasts are part of the multiply-add and four steps are staged at once, and the
entries of dJ/dA are shared by 64/N groups of lanes, evenly (2, 16) or not (5, 13).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 5, 9, 10, 13, 16, 17, 24])
@pytest.mark.parametrize("tableau", ["TAB_CASH_KARP54", "TAB_DOPRI5"])
def test_long_instances_match_oracle(n, tableau):
    import torch
    import oracle as O
    import vectorizedadjoint_amd as va
    assert torch.cuda.is_available(), "no HIP device"
    B = 150
    rng = np.random.default_rng(n)
    # a stable community: stiffness bounds the steps, so their number follows the
    # rates, from tens to some 1,500
    r = rng.uniform(0.05, 2.0, (1, B)) * rng.uniform(0.9, 1.1, (n, B))
    A = 0.3 / n * rng.uniform(-1.0, 1.0, (n, n, B))
    A[np.arange(n), np.arange(n)] = -1.0
    p = np.concatenate([r, A.reshape(n * n, B)])
    y0 = rng.uniform(0.2, 0.8, (n, B))
    kw = dict(t1=2000.0, dt0=1e-3, abs_tol=1e-8, rel_tol=1e-8, max_steps=8192)
    tab = getattr(va, tableau)
    o = O.solve_batch(O.problem(va.SYS_LOTKA_VOLTERRA, n, n + n * n, tab, controlled=True, **kw),
                      y0, p, va.COST_SUM, nthreads=8)
    pb = va.Problem(system=va.SYS_LOTKA_VOLTERRA, n_state=n, n_param=n + n * n, batch=B,
                    tableau=tab, adaptive=True, lanes=64, block_size=64, **kw)
    att = o["n_acc"] + o["n_rej"]
    assert (o["status"] == 0).all() and (o["n_acc"] >= 256).sum() >= 8 and (att >= 448).sum() >= 8
    print(f"[gpu] long reverse N={n} {tableau}, attempts {att.min()}..{att.max()}", flush=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    with va.Solver(pb) as s:
        for _ in range(2):
            out = s.solve(dev(y0), dev(p), va.COST_SUM)
            torch.cuda.synchronize()
            for k in ("n_acc", "yT", "J", "dJdy0", "dJdp"):
                g = out[k].cpu().numpy()
                assert np.array_equal(g, o[k]), (k, n)
