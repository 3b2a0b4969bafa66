"""Which Lotka-Volterra reverses of several seeds take them in turn, CPU only: large
batches of few species, but where the seeds of a few instances fill a wave."""
import pytest

import launches as L
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


def _system(n, **kw):
    return dict(system=K.SYS_LOTKA_VOLTERRA, n=n, np=n + n * n, **kw)


# by N the numbers of seeds that large batches take in turn, of those called
IN_TURN = {2: {2, 3}, 3: {2, 3}, 4: {2, 3}, 5: {5}, 6: {3, 6}, 7: {2, 7}, 8: set(), 10: set()}


@pytest.mark.parametrize("n", IN_TURN)
def test_seeds_of_large_batches_in_turn(exe, n):
    for batch in (32768, 32769):
        ops = {"adjoint:1": 1, "adjoint:2": 2, "adjoint:3": 3, "sens": n, "solve": 1}
        calls = L.log(exe, ["forward", *ops],
                      **_system(n, tableau=K.TAB_CASH_KARP54, batch=batch, occupancy=4))
        for (op, seeds), call in zip(ops.items(), calls[1:]):
            for l in call:
                if l.kernel.startswith("k_glv_rows_rev<"):
                    want = batch > 32768 and seeds in IN_TURN[n]
                    assert l["in_turn"] == str(int(want)), (op, l)
