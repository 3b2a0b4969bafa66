"""Reverses without a long-instance kernel beside them: the head of their order
(instances of 256 and more accepted steps) in blocks of three waves, for every way in
which those waves hold an instance, against the oracle, bit for bit: a solve, and one
seed through adjoint() that adds to mu.  The instances past half of the grid's blocks
and the short ones take the ordinary sweep of the same launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# N=2..16 sweep the head so; the entries of dJ/dA are shared by 64/N groups of lanes,
# evenly (2, 4, 8, 16) or not
SIZES = [2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("tableau", ["TAB_CASH_KARP54", "TAB_DOPRI5", "TAB_FEHLBERG78"])
def test_head_of_the_order_matches_oracle(n, tableau):
    import torch
    import oracle as O
    import vectorizedadjoint_amd as va
    assert torch.cuda.is_available(), "no HIP device"
    B = 600
    rng = np.random.default_rng(100 + n)
    # a stable community: stiffness bounds the steps, so their number follows the rates
    r = np.exp(rng.uniform(np.log(0.02), np.log(2.0), (1, B))) * rng.uniform(0.9, 1.1, (n, B))
    A = 0.3 / n * rng.uniform(-1.0, 1.0, (n, n, B))
    A[np.arange(n), np.arange(n)] = -1.0
    p = np.concatenate([r, A.reshape(n * n, B)])
    y0 = rng.uniform(0.2, 0.8, (n, B))
    kw = dict(t1=1000.0, dt0=1e-3, abs_tol=1e-8, rel_tol=1e-8, max_steps=4096)
    tab = getattr(va, tableau)
    o = O.solve_batch(O.problem(va.SYS_LOTKA_VOLTERRA, n, n + n * n, tab, controlled=True, **kw),
                      y0, p, va.COST_SUM, nthreads=8)
    assert (o["status"] == 0).all()
    blocks = -(-B // (4 * (64 // n)))  # of the reverse's grid
    long = int((o["n_acc"] >= 256).sum())
    assert long >= 8 and blocks >= 4 and (o["n_acc"] < 200).any(), (long, blocks)
    print(f"[gpu] head of the reverse N={n} {tableau}: {long} long, {blocks} blocks", flush=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    pb = va.Problem(system=va.SYS_LOTKA_VOLTERRA, n_state=n, n_param=n + n * n, batch=B,
                    tableau=tab, adaptive=True, **kw)
    with va.Solver(pb) as s:
        out = s.solve(dev(y0), dev(p), va.COST_SUM)
        torch.cuda.synchronize()
        for k in ("n_acc", "yT", "J", "dJdy0", "dJdp"):
            assert np.array_equal(out[k].cpu().numpy(), o[k]), (k, n)
        s.forward(dev(y0), dev(p))
        mu0 = rng.normal(size=(1, n + n * n, B))
        lam, mu = s.adjoint(dev(p), torch.ones((1, n, B), dtype=torch.float64).cuda(), dev(mu0))
        torch.cuda.synchronize()
        assert np.array_equal(lam.cpu().numpy()[0], o["dJdy0"])
        assert np.array_equal(mu.cpu().numpy()[0], mu0[0] + o["dJdp"])
