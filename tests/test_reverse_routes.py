"""Which reverse kernel a Lotka-Volterra call takes, CPU only: the blocks of three waves
for the head of the order (the HEAD instantiation with part 2) in one-seed reverses of
up to 16 species, adaptive, in blocks of 256 threads, and nowhere else."""
import pytest

import codeobjects
import launches as L
import vectorizedadjoint_amd as va
from vectorizedadjoint_amd import constants as K


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return L.build(tmp_path_factory.mktemp("launches"))


@pytest.mark.parametrize("n", range(2, 33))
def test_head_blocks_of_one_seed_reverses(exe, n):
    for tableau, adaptive in ((K.TAB_CASH_KARP54, 1), (K.TAB_DOPRI5, 1), (K.TAB_FEHLBERG78, 1),
                              (K.TAB_RK4, 0)):
        calls = L.log(exe, ["solve", "forward", "adjoint:1", "adjoint:2", "sens"],
                      system=K.SYS_LOTKA_VOLTERRA, n=n, np=n + n * n, tableau=tableau,
                      adaptive=adaptive, batch=600)
        head = n <= 16 and adaptive
        for op, call in zip(("solve", "forward", "adjoint:1", "adjoint:2", "sens"), calls):
            revs = [l for l in call if l.kernel.startswith("k_glv_rows_rev<")]
            assert len(revs) == (op != "forward"), (op, call)
            for l in revs:
                one = op in ("solve", "adjoint:1")
                assert (l["part"] == "2") == (head and one), (op, l)
                assert l["items"] == {"adjoint:2": "2", "sens": str(n)}.get(op, "1")


@pytest.mark.parametrize("n", (2, 3, 5, 10, 13, 16, 17))
def test_reverses_without_a_head_are_not_held_to_its_registers(exe, n):
    """The variant with a head serves every reverse but where it holds fewer blocks per
    CU than the sweep alone."""
    ks = codeobjects.kernels(va.library_path())
    blocks = lambda k: 512 // ((k[".vgpr_count"] + 7) // 8 * 8)  # of a wave per SIMD
    system = dict(system=K.SYS_LOTKA_VOLTERRA, n=n, np=n + n * n, batch=600)
    for tableau in (K.TAB_CASH_KARP54, K.TAB_DOPRI5, K.TAB_FEHLBERG78):
        # few lanes: from the second solve on beside the long-instance kernel, for N=10
        for lanes in (0, 30):
            for call in L.log(exe, ["solve", "solve", "forward", "adjoint:1", "adjoint:2", "sens"],
                              tableau=tableau, lanes=lanes, **system):
                for l in call:
                    if not l.kernel.startswith("k_glv_rows_rev<"):
                        continue
                    lean = n == 2 and tableau == K.TAB_FEHLBERG78 and l["part"] != "2"
                    assert l.kernel.endswith("true>") == (n <= 16 and not lean), l
                    if lean:
                        head = l.kernel.replace("false>", "true>")
                        assert blocks(ks[l.kernel]) > blocks(ks[head])
