"""The kernels for waves that run alone (constants in vector registers), CPU only: none
of them keeps values in scratch memory, which costs more than the constants save,
and the launch rule takes them only where they exist and waves have a SIMD each."""
import pytest

import codeobjects
import launches as L
import vectorizedadjoint_amd as va
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


def _is_lone(name):
    args = [a.strip() for a in name[name.index("<") + 1:name.rindex(">")].split(",")] \
        if "<" in name else []
    return (name.startswith("k_fwd<") and args[-2] == "true") or \
           (name.startswith("k_rev<") and args[-2] == "true") or \
           (name.startswith(("k_obs_fwd<", "k_obs_rev<")) and args[-1] == "true")


def test_no_lone_kernel_uses_scratch_memory():
    ks = {n: k for n, k in codeobjects.kernels(va.library_path()).items() if _is_lone(n)}
    assert len(ks) > 50
    bad = {n: k[".private_segment_fixed_size"] for n, k in ks.items()
           if k[".private_segment_fixed_size"]}
    assert not bad, bad


@pytest.mark.parametrize("system,n,np,ipw", [(K.SYS_VAN_DER_POL, 2, 1, 0),
                                             (K.SYS_LOTKA_VOLTERRA, 3, 12, 64),
                                             (K.SYS_LOTKA_VOLTERRA, 4, 20, 64),
                                             (K.SYS_LOTKA_VOLTERRA, 5, 30, 64)])
@pytest.mark.parametrize("tableau", [K.TAB_CASH_KARP54, K.TAB_DOPRI5, K.TAB_FEHLBERG78])
def test_launches_take_lone_kernels_up_to_a_wave_per_simd(exe, system, n, np, ipw, tableau):
    for batch, lone in ((1, True), (65536, True), (65537, False)):
        calls = L.log(exe, ["forward", "adjoint:1", "adjoint:2"], system=system, n=n, np=np,
                      tableau=tableau, batch=batch, ipw=ipw)
        fwd, = [l for l in calls[0] if l.kernel.startswith("k_fwd")]
        assert _is_lone(fwd.kernel) == (lone and n <= 4)
        spills = n == 4 and tableau == K.TAB_FEHLBERG78
        for call, seeds in ((calls[1], 1), (calls[2], 2)):
            rev, = [l for l in call if l.kernel.startswith("k_rev")]
            threads = int(rev["grid"]) * int(rev["block"])
            want = threads <= 65536 and n <= 4 and not spills
            assert _is_lone(rev.kernel) == want, (batch, seeds, rev)
