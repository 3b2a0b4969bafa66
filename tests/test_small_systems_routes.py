"""Which layout Lotka-Volterra forwards of few species and of fixed steps take, CPU only:
one instance per 16-lane row only up to the batches where that is the faster layout."""
import pytest

import launches as L
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


def _system(n, **kw):
    return dict(system=K.SYS_LOTKA_VOLTERRA, n=n, np=n + n * n, **kw)


@pytest.mark.parametrize("tableau,adaptive,most", [
    (K.TAB_CASH_KARP54, 1, {2: 0, 3: 1024, 4: 1024, 5: 8192, 7: 8192, 13: 8192}),
    (K.TAB_FEHLBERG78, 1, {2: 0, 3: 1024, 6: 8192, 8: 8192}),
    (K.TAB_RK4, 0, {2: 0, 3: 4096, 5: 4096, 7: 4096, 10: 4096, 16: 4096}),
])
def test_forward_layout(exe, tableau, adaptive, most):
    for n, rows in most.items():
        for batch in (1, rows, rows + 1):
            if batch < 1:
                continue
            call, = L.log(exe, ["forward"], **_system(n, tableau=tableau, adaptive=adaptive,
                                                      batch=batch, occupancy=2))
            fwd, = [l for l in call if l.kernel.startswith("k_glv_rows_fwd")]
            # in index order adaptive batches of 10 and more species keep it
            want = batch <= rows or (adaptive and n >= 10)
            assert ("(Lay)1" in fwd.kernel) == want, (n, batch, fwd)
