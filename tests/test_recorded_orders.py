"""Which buffer each launch of a handle takes its instance order from, CPU only (the
launches are logged, not run).  A solve that a caller records into a graph does not
run when it is enqueued: the next eager solve must not take an order that only the
recording would have written, and a replay must read the order that the one before
it left."""
import pytest

import launches as L
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


HANDLES = {
    "vdp": dict(system=K.SYS_VAN_DER_POL, n=2, np=1, tableau=K.TAB_DOPRI5, batch=1000),
    "vdp tiled": dict(system=K.SYS_VAN_DER_POL, n=2, np=1, tableau=K.TAB_DOPRI5, batch=5000),
    "vdp observed": dict(system=K.SYS_VAN_DER_POL, n=2, np=1, tableau=K.TAB_DOPRI5, batch=1000,
                         n_obs=4),
    "vdp checkpoints": dict(system=K.SYS_VAN_DER_POL, n=2, np=1, tableau=K.TAB_DOPRI5,
                            batch=1000, n_obs=4, slots=2),
    "glv10 split": dict(system=K.SYS_LOTKA_VOLTERRA, n=10, np=110, tableau=K.TAB_CASH_KARP54,
                        batch=2000, lanes=120),
    "glv5": dict(system=K.SYS_LOTKA_VOLTERRA, n=5, np=30, tableau=K.TAB_CASH_KARP54, batch=2000,
                 lanes=120),
}


def _op(name):
    return "observed" if HANDLES[name].get("n_obs") else "solve"


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("before", [0, 1, 2, 3])
def test_no_order_is_taken_that_only_a_recording_writes(exe, name, before):
    op = _op(name)
    ops = [op] * before + ["capture", op, op, "end", op, op, op]
    calls = L.log(exe, ops, **HANDLES[name])
    launched = [l for c in calls for l in c]
    assert any(l.recorded for l in launched)
    bad = [l for l in launched if l.unwritten]
    assert not bad, bad


def _forwards(call):
    return [l for l in call if l.kernel.startswith(("k_fwd", "k_obs_fwd", "k_glv_rows"))
            and "rev" not in l.kernel]


@pytest.mark.parametrize("name", HANDLES)
def test_a_replay_reads_the_order_the_one_before_left(exe, name):
    op = _op(name)
    calls = L.log(exe, [op, op, "capture", op, "end"], **HANDLES[name])
    recorded = calls[3]
    assert all(l.recorded for l in recorded)
    taken = {l["order"] for l in _forwards(recorded)}
    left = {l["out1"] for l in recorded if "out1" in l.fields}
    assert taken == left and len(taken) == 1, (taken, left)


def test_an_adjoint_after_a_recorded_forward_has_an_order(exe):
    calls = L.log(exe, ["capture", "forward", "end", "adjoint:1", "adjoint:2", "sens"],
                  **HANDLES["vdp tiled"])
    assert not [l for c in calls for l in c if l.unwritten]
