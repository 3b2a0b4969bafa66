"""Reverse sweeps of several seeds against the same seeds swept one call at a time.

A seed's sweep is the same operations whether its lane holds it alone, beside a
second seed or in turn with the others, and whichever kernel takes the instance,
so the results are compared bit for bit.  The one-seed sweep itself is compared
with the oracle in test_gpu_parity.py.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.cpu().numpy().view(np.int64)


def _solver(system, B, **kw):
    import torch
    import vectorizedadjoint_amd as va
    from vectorizedadjoint_amd import inputs as I
    assert torch.cuda.is_available(), "no HIP device"
    w = I.WORKLOADS[system]
    inp = I.make_inputs(w, B)
    s = va.Solver(va.Problem.from_workload(w, batch=B, max_steps=1024, **kw))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return torch, s, dev(inp["y0"]), dev(inp["p"])


# Van der Pol: up to 65536 (instance, seed) pairs each seed has a lane of its own,
# above that a lane takes two (an odd count leaves one alone); glv10 with few lanes:
# index order, then the split schedule with its one-wave sweeps of long instances.
@pytest.mark.parametrize("system,B,nout,kw", [
    ("vdp", 1, 2, {}), ("vdp", 70, 3, {}), ("vdp", 22000, 3, {"t1": 2.0}),
    ("vdp", 40000, 2, {"t1": 2.0}), ("vdp", 300, 5, {"lanes": 64, "block_size": 64}),
    ("glv10", 130, 4, {"t1": 10.0}), ("glv10", 1500, 2, {"lanes": 120, "block_size": 64}),
])
def test_seeds_together_match_one_by_one(system, B, nout, kw):
    torch, s, y0, p = _solver(system, B, **kw)
    n, P = y0.shape[0], p.shape[0]
    print(f"[gpu] {nout} seeds {system} B={B} {kw}", flush=True)
    g = torch.Generator().manual_seed(7)
    lam0 = torch.randn((nout, n, B), generator=g, dtype=torch.float64).cuda()
    mu0 = torch.randn((nout, P, B), generator=g, dtype=torch.float64).cuda()
    with s:
        for _ in range(2):  # index order, then the order the first forward left
            s.forward(y0.clone(), p)
            lam, mu = s.adjoint(p, lam0.clone(), mu0.clone())
            for o in range(nout):
                l1, m1 = s.adjoint(p, lam0[o:o + 1].clone(), mu0[o:o + 1].clone())
                assert np.array_equal(_bits(lam[o]), _bits(l1[0]))
                assert np.array_equal(_bits(mu[o]), _bits(m1[0]))


@pytest.mark.parametrize("system,B,kw", [
    ("vdp", 65, {}), ("vdp", 33000, {"t1": 2.0}), ("glv10", 90, {"t1": 10.0}),
    ("glv10", 1500, {"lanes": 120, "block_size": 64, "max_attempts": 500}),
])
def test_sensitivity_matrix_matches_unit_seeds(system, B, kw):
    """The matrix against unit seeds through adjoint(); failed instances are NaN."""
    torch, s, y0, p = _solver(system, B, **kw)
    n, P = y0.shape[0], p.shape[0]
    print(f"[gpu] sensitivity {system} B={B} {kw}", flush=True)
    with s:
        for _ in range(2):
            s.forward(y0.clone(), p)
            S = s.sensitivity_matrix(p)
            lam = torch.eye(n, dtype=torch.float64).cuda()[:, :, None].expand(n, n, B).contiguous()
            mu = torch.zeros((n, P, B), dtype=torch.float64).cuda()
            s.adjoint(p, lam, mu)
            assert np.array_equal(_bits(torch.isnan(S).double()), _bits(torch.isnan(mu).double()))
            assert np.array_equal(_bits(S.nan_to_num()), _bits(mu.nan_to_num()))
