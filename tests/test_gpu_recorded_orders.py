"""Solves recorded by the caller (torch.cuda.graph) on handles that reuse an instance
order: an eager solve between the recording and its first replay, and replays on new
data with eager solves between them, give a fresh handle's results bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,B,lanes", [("vdp", 1000, 0), ("vdp", 4161, 0),
                                          ("vdp_obs", 700, 0), ("glv10", 1024, 120)])
def test_eager_solves_beside_a_recorded_one(name, B, lanes):
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    w = I.WORKLOADS[name]
    kw = dict(batch=B, max_steps=1024, lanes=lanes)
    obs = ()
    if name == "vdp_obs":
        kw.update(n_obs=5, checkpoint_slots=8, t1=2.0)
        t = torch.linspace(0.4, 2.0, 5, dtype=torch.float64).cuda()
        obs = t, torch.stack([t.cos(), t.sin()], dim=1).contiguous()
    pb = va.Problem.from_workload(w, **kw)
    inp = I.make_inputs(w, 4 * B)
    data = [tuple(torch.from_numpy(inp[k][:, i::4].copy()).cuda() for k in ("y0", "p"))
            for i in range(4)]
    y0, p = data[0][0].clone(), data[0][1].clone()
    print(f"[gpu] recorded solve {name} B={B} lanes={lanes}", flush=True)

    def call(s, out=None):
        return s.solve_observed(y0, p, *obs, out=out) if obs else s.solve(y0, p, w.cost, out=out)

    def same(a):
        with va.Solver(pb) as fresh:
            b = call(fresh)
            torch.cuda.synchronize()
            for k in a:
                assert torch.equal(a[k].nan_to_num(7.0), b[k].nan_to_num(7.0)), k

    with va.Solver(pb) as s:
        out = call(s)  # one eager solve: the only order there is
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call(s, out)
        for v in out.values():
            v.zero_()
        same(call(s))  # before any replay
        for y, q in data:
            y0.copy_(y)
            p.copy_(q)
            for v in out.values():
                v.zero_()
            g.replay()
            torch.cuda.synchronize()
            same(out)
            same(call(s))
