"""Full-chip launches of the two-state one-lane kernels (more than 65,536 lanes): rows
stored and read by lines of four.  The same instances solved in a small batch, whose
kernels store and load each row by its own lane, give the same bits; the oracle
covers those in test_gpu_parity.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(w, inp, cols, solves, **kw):
    import torch
    import vectorizedadjoint_amd as va
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a[:, cols])).cuda()
    y0, p = dev(inp["y0"]), dev(inp["p"])
    with va.Solver(va.Problem.from_workload(w, batch=y0.shape[1], **kw)) as s:
        for _ in range(solves):
            out = s.solve(y0, p, w.cost)
        out["digest"] = s.step_digest()
        rows = [s.trajectory(b) for b in (0, 1)]
        torch.cuda.synchronize()
        return {k: v.cpu().numpy() for k, v in out.items()}, rows


# the tail of the batch is a partial tile; t1 makes step counts short, with every
# remainder of four rows, zero steps (t1 = t0) and instances that meet the step cap
@pytest.mark.parametrize("name,B,kw", [
    ("vdp", 65793, {"t1": 0.5, "max_steps": 256}),
    ("vdp", 70000, {"t1": 1.0, "max_steps": 60}),
    ("oscillator", 131072 + 5, {"t1": 0.3, "max_steps": 256}),
    ("oscillator", 66000, {"t1": 0.0, "max_steps": 4}),
    ("vdp", 66000, {"t1": 0.5, "max_steps": 256, "block_size": 64}),
])
def test_lines_match_rows(name, B, kw):
    import torch
    from vectorizedadjoint_amd import inputs as I
    assert torch.cuda.is_available(), "no HIP device"
    w = I.WORKLOADS[name]
    inp = I.make_inputs(w, B)
    print(f"[gpu] lines {name} B={B} {kw}", flush=True)
    few = np.r_[0:300, B - 300:B]
    for solves in (1, 2):  # index order, then longest first
        big, rows = _solve(w, inp, slice(None), solves, **kw)
        small, srows = _solve(w, inp, few, 1, **kw)
        assert big["n_acc"].max() - big["n_acc"].min() >= (0 if kw["t1"] == 0.0 else 4)
        for k in small:
            a, b = big[k][..., few], small[k]
            assert np.array_equal(a.view(np.int64) if a.dtype == np.float64 else a,
                                  b.view(np.int64) if b.dtype == np.float64 else b), k
        for a, b in zip(rows, srows):
            assert np.array_equal(a, b)


def test_adjoint_adds_to_mu_by_lines():
    """One seed through adjoint() (mu += dJ/dp) on a full chip, against a small batch."""
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    w = I.WORKLOADS["oscillator"]
    B = 66001
    inp = I.make_inputs(w, B)
    few = np.r_[0:100, B - 100:B]
    res = []
    for cols in (slice(None), few):
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a[:, cols])).cuda()
        y0, p = dev(inp["y0"]), dev(inp["p"])
        n = y0.shape[1]
        with va.Solver(va.Problem.from_workload(w, batch=n, t1=0.3, max_steps=256)) as s:
            s.forward(y0, p)
            lam = torch.ones((1, 2, n), dtype=torch.float64).cuda() * 0.5
            mu = torch.full((1, 2, n), 3.0, dtype=torch.float64).cuda()
            s.adjoint(p, lam, mu)
            res.append((lam.cpu().numpy(), mu.cpu().numpy()))
    assert np.array_equal(res[0][0][..., few], res[1][0])
    assert np.array_equal(res[0][1][..., few], res[1][1])
