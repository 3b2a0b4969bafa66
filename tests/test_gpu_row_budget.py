"""Tiled and instance-major row stores of one batch: a trajectory budget of the rows
alone has no room for whole tiles, so the handle keeps its rows instance-major; without
a budget they are tiled.  Results and stored rows are the same, and the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,max_steps", [(4096, 2045), (4161, 2047)])
def test_tiled_and_instance_major_stores_agree(B, max_steps):
    import torch
    import oracle as O
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    assert torch.cuda.is_available(), "no HIP device"
    w = I.WORKLOADS["vdp"]
    inp = I.make_inputs(w, B)
    opb = O.problem(w.system, w.n, w.np, w.tableau, t0=w.t0, t1=w.t1, dt0=w.dt0, abs_tol=w.tol,
                    rel_tol=w.tol, max_steps=max_steps)
    y0, p = torch.from_numpy(inp["y0"]).cuda(), torch.from_numpy(inp["p"]).cuda()
    exact = 8 * B * (max_steps + 1) * (w.n + 2)
    outs, rows = [], []
    for budget in (0, exact):
        print(f"[gpu] row store B={B} max_steps={max_steps} budget={budget}", flush=True)
        with va.Solver(va.Problem.from_workload(w, batch=B, max_steps=max_steps,
                                                trajectory_budget_bytes=budget)) as s:
            for _ in range(2):  # index order, then longest first
                out = s.solve(y0, p, w.cost)
                torch.cuda.synchronize()
                outs.append({k: v.cpu().numpy() for k, v in out.items()})
                rows.append([s.trajectory(b) for b in (0, 63, 64, B - 1)])
    for o, r in zip(outs[1:], rows[1:]):
        for k in o:
            assert np.array_equal(outs[0][k], o[k], equal_nan=True), k
        assert all(np.array_equal(x, y) for x, y in zip(rows[0], r))
    for b, r in zip((0, 63, 64, B - 1), rows[0]):
        o = O.Solve(opb, inp["y0"][:, b].copy(), inp["p"][:, b].copy())
        assert np.array_equal(r[:, 0], o.times) and np.array_equal(r[:, 2:], o.states)
