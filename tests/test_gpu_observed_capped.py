"""Observed solves with checkpoints after a solve that ran out of steps: with
max_steps and the slots powers of two, instances that ended at the cap (MAX_STEPS)
give the next solve on the handle its starting spacing, and that solve, under
parameters with which the same instances end OK in more than stride_max steps,
gives a fresh handle's results bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block,levels", [(256, 1), (64, 1), (256, 2)])
def test_solve_after_one_that_ran_out_of_steps(block, levels):
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    B, K, cap, slots = 512, 12, 1024, 8
    stride_max = cap // slots
    w = I.WORKLOADS["vdp_obs"]
    inp = I.make_inputs(w, B)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    y0 = dev(inp["y0"])
    stiff, mild = dev(np.full((1, B), 100.0)), dev(np.linspace(0.5, 5.0, B)[None])
    t_obs = 12.0 * np.arange(1, K + 1) / K
    y_obs = np.stack([2 * np.cos(t_obs), -2 * np.sin(t_obs)], axis=1)
    pb = va.Problem.from_workload(w, batch=B, t1=12.0, n_obs=K, max_steps=cap,
                                  checkpoint_slots=slots, block_size=block,
                                  flags=va.FLAG_CHECKPOINT_2LEVEL if levels == 2 else 0)
    print(f"[gpu] observed after MAX_STEPS B={B} block={block} levels={levels}", flush=True)
    with va.Solver(pb) as used, va.Solver(pb) as fresh:
        o = dev(t_obs), dev(y_obs)
        for _ in range(2):  # the second in the order that the first left
            first = used.solve_observed(y0, stiff, *o)
        a = used.solve_observed(y0, mild, *o)
        b = fresh.solve_observed(y0, mild, *o)
        torch.cuda.synchronize()
        # the premise: at the cap before, above stride_max and OK now
        assert (first["status"] != 0).any() and int(first["n_acc"].max()) == cap
        assert (a["status"] == 0).all() and int(a["n_acc"].max()) > stride_max
        for k in a:
            assert torch.equal(a[k], b[k]), k
