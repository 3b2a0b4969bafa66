"""From how many attempts the long instances of a Lotka-Volterra solve are taken by
their own kernel, CPU only: the higher count is for batches that fill the device, which
a caller's smaller number of lanes does not make of a batch."""
import pytest

import launches as L
from vectorizedadjoint_amd import constants as K

GLV10 = dict(system=K.SYS_LOTKA_VOLTERRA, n=10, np=110, tableau=K.TAB_CASH_KARP54, occupancy=2)
FULL = 2 * 256 * 24  # blocks per CU x CUs x instances of a block (four waves of six)


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


@pytest.mark.parametrize("batch,lanes,bucket", [
    (5 * FULL // 3, 0, 32), (5 * FULL // 3 + 1, 0, 56),
    (2000, 120, 32), (5 * FULL // 3, 120, 32), (5 * FULL // 3 + 1, 120, 56)])
def test_long_set_by_the_device_not_by_the_lanes(exe, batch, lanes, bucket):
    calls = L.log(exe, ["solve", "solve", "forward"], batch=batch, lanes=lanes, **GLV10)
    for call in calls:
        scatter, = [l for l in call if l.kernel == "k_order_scatter"]
        assert scatter["long1"] == str(bucket), scatter
