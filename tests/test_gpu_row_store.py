"""The tiled row store of the one-lane kernels: an instance's rows read back through
trajectory() against the oracle's stored points, after an index-order forward (slot
b is instance b's) and after an ordered one (the k-th instance taken is in slot k),
at batches around a tile of 64 slots and step counts around a block of 4 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,max_steps", [(1, 2048), (63, 2048), (65, 2047), (130, 2046)])
def test_rows_match_oracle_in_either_order(B, max_steps):
    import torch
    import oracle as O
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    assert torch.cuda.is_available(), "no HIP device"
    w = I.WORKLOADS["vdp"]
    inp = I.make_inputs(w, B)
    pb = O.problem(w.system, w.n, w.np, w.tableau, t0=w.t0, t1=w.t1, dt0=w.dt0, abs_tol=w.tol,
                   rel_tol=w.tol, max_steps=max_steps)
    print(f"[gpu] row store B={B} max_steps={max_steps}", flush=True)
    y0, p = torch.from_numpy(inp["y0"]).cuda(), torch.from_numpy(inp["p"]).cuda()
    with va.Solver(va.Problem.from_workload(w, batch=B, max_steps=max_steps)) as s:
        for _ in range(2):
            s.forward(y0.clone(), p)
            for b in sorted({0, B // 2, B - 1}):
                o = O.Solve(pb, inp["y0"][:, b].copy(), inp["p"][:, b].copy())
                rows = s.trajectory(b)
                assert np.array_equal(rows[:, 0], o.times)
                assert np.array_equal(rows[:-1, 1], np.diff(o.times))
                assert np.array_equal(rows[:, 2:], o.states)


def test_failed_instances_rows_end_at_their_last_step():
    """A step cap that every instance meets: cap rows are stored, none beyond."""
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    w = I.WORKLOADS["vdp"]
    inp = I.make_inputs(w, 70)
    y0, p = torch.from_numpy(inp["y0"]).cuda(), torch.from_numpy(inp["p"]).cuda()
    with va.Solver(va.Problem.from_workload(w, batch=70, max_steps=5)) as s, \
            va.Solver(va.Problem.from_workload(w, batch=70, max_steps=2048)) as full:
        s.forward(y0.clone(), p)
        full.forward(y0.clone(), p)
        for b in (0, 63, 64, 69):
            assert np.array_equal(s.trajectory(b), full.trajectory(b)[:5])
