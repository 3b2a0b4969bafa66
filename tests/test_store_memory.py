"""How much device memory a handle's store needs, CPU only: a batch that fits as plain
rows is accepted on any device with that much or more, whatever the tiled rows and
their slots would take beyond it."""
import os
import subprocess

import pytest

import launches as L
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


@pytest.mark.parametrize("batch,n_obs", [(4096, 0), (4100, 0), (5000, 3)])
def test_more_memory_never_refuses_what_less_accepts(exe, batch, n_obs):
    args = [K.SYS_VAN_DER_POL, 2, 1, K.TAB_DOPRI5, 1, batch, 0, 0, n_obs, 0, 0, 2]
    plain = batch * 9 * 4 * 8  # max_steps 8: rows 0..8 of four doubles
    tiled = (batch + 63) // 64 * 64 * 12 * 4 * 8

    def accepted(memory):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True,
                           env=dict(os.environ, LAUNCH_LOG_MEMORY=str(memory)))
        assert r.returncode in (0, 1), r.stderr
        return r.returncode == 0

    step = batch * 2  # half of an array of counts
    got = [accepted(m) for m in range(plain, tiled + batch * 4 * (8 + n_obs) + 8192, step)]
    assert not got[0] and got[-1]
    first = got.index(True)
    assert all(got[first:]), [plain + k * step for k in range(first, len(got)) if not got[k]]
