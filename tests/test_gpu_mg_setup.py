"""A multigrid set-up that fails (a non-finite field) leaves no trace: on the
other members of an ensemble, nor on the handle itself once its field is
repaired."""
import numpy as np
import pytest

from . import scenarios as S

pytestmark = pytest.mark.gpu

SIZES = [(9, 9, 9), (12, 10, 11), (17, 9, 13), (10, 11, 19)]


def _bad_modulus(s):
    E = s["E_elem"].copy()
    E[E.size // 2] = np.nan
    return E


def _start(s):
    return np.zeros(3 * int(np.prod(s["n"])))


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("bad", [0, 2], ids=["first", "middle"])
def test_batch_set_up_failure_leaves_no_trace(bad, mixed):
    """Every member, solved again after the bad one is repaired, gives what it
    gives alone on a fresh handle (bitwise, as any member of a mix), in the
    batch and in a solve of its own."""
    from vpfhf_amd import VfgError, _lib
    from vpfhf_amd.batch import Batch
    sc = [S.make(n=n, seed=11 + i, nu=0.3) for i, n in enumerate(SIZES)]
    Z = [_start(s) for s in sc]
    ref, solo = [], []
    for s, z in zip(sc, Z):
        P = S.to_gpu(s)
        B = Batch([P])
        ref.append(B.u_solve([z], [z], mixed=mixed, pc=_lib.PC_MG)[0][0])
        B.close()
        P.close()
        P = S.to_gpu(s)
        solo.append(P.VF_StepU(z, z)[0])
        P.close()
    Ps = [S.to_gpu(s) for s in sc]
    Ps[bad].set_fields(E_elem=_bad_modulus(sc[bad]))
    B = Batch(Ps)
    with pytest.raises(VfgError):
        B.u_solve(Z, Z, mixed=mixed, pc=_lib.PC_MG)
    Ps[bad].set_fields(E_elem=sc[bad]["E_elem"])
    U, infos = B.u_solve(Z, Z, mixed=mixed, pc=_lib.PC_MG)
    assert all(i.status == 0 for i in infos)
    for u, r in zip(U, ref):
        assert np.array_equal(u, r)
    B.close()
    for P, z, r in zip(Ps, Z, solo):
        u, info = P.VF_StepU(z, z)
        assert info.status == 0 and np.array_equal(u, r)
        P.close()


def test_set_up_failure_is_repaired_with_the_field():
    from vpfhf_amd import VfgError
    s = S.make(n=(17, 9, 13), seed=5, nu=0.3)
    z = _start(s)
    P = S.to_gpu(s)
    ref = P.VF_StepU(z, z)[0]
    P.close()
    P = S.to_gpu(s)
    P.set_fields(E_elem=_bad_modulus(s))
    with pytest.raises(VfgError):
        P.VF_StepU(z, z)
    P.set_fields(E_elem=s["E_elem"])
    u, info = P.VF_StepU(z, z)
    assert info.status == 0 and np.array_equal(u, ref)
    P.close()
