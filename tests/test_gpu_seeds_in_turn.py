"""Several seeds of batches whose instances may take them in turn, against the same
seeds swept one call at a time, bit for bit: with no long instance (in turn), with some
(items of one seed), and at the batch where the rule starts."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.cpu().numpy().view(np.int64)


@pytest.mark.parametrize("n,B,t1,nout,long", [
    (2, 32768, 4.0, 2, False), (2, 32769, 4.0, 2, False), (2, 33000, 4.0, 5, False),
    (3, 33001, 4.0, 3, False), (5, 40003, 4.0, 2, False), (7, 33000, 4.0, 3, False),
    (5, 33000, 60.0, 2, True), (8, 33000, 4.0, 2, False),
])
def test_seeds_match_one_by_one(n, B, t1, nout, long):
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    assert torch.cuda.is_available(), "no HIP device"
    w = dataclasses.replace(I.WORKLOADS["glv10"], n=n, np=n + n * n, t1=t1)
    inp = I.make_inputs(w, B)
    y0, p = (torch.from_numpy(inp[k]).cuda() for k in ("y0", "p"))
    g = torch.Generator().manual_seed(n)
    lam0 = torch.randn((nout, n, B), generator=g, dtype=torch.float64).cuda()
    mu0 = torch.randn((nout, n + n * n, B), generator=g, dtype=torch.float64).cuda()
    n_acc = torch.empty(B, dtype=torch.int32, device="cuda")
    status = torch.empty(B, dtype=torch.int32, device="cuda")
    print(f"[gpu] {nout} seeds N={n} B={B} t1={t1}", flush=True)
    with va.Solver(va.Problem.from_workload(w, batch=B, max_steps=768)) as s:
        s.forward(y0.clone(), p, n_accepted=n_acc, lane_status=status)
        assert bool((n_acc[status == 0] >= 256).any()) == long
        lam, mu = s.adjoint(p, lam0.clone(), mu0.clone())
        for o in range(nout):
            l1, m1 = s.adjoint(p, lam0[o:o + 1].clone(), mu0[o:o + 1].clone())
            assert np.array_equal(_bits(lam[o].nan_to_num()), _bits(l1[0].nan_to_num()))
            assert np.array_equal(_bits(mu[o].nan_to_num()), _bits(m1[0].nan_to_num()))
        S = s.sensitivity_matrix(p)
        for o in range(n):
            e = torch.zeros((1, n, B), dtype=torch.float64, device="cuda")
            e[0, o] = 1.0
            m = torch.zeros((1, n + n * n, B), dtype=torch.float64, device="cuda")
            s.adjoint(p, e, m)
            assert np.array_equal(_bits(S[o].nan_to_num()), _bits(m[0].nan_to_num()))
