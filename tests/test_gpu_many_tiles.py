"""Grids of more workgroup tiles than the solvers keep reduction partials for:
long bars of one element in y and z, one 15-node tile per 15 nodes.  The
products and the post-smoothing then reduce in a pass of their own."""
import numpy as np
import pytest

from . import scenarios as S

pytestmark = pytest.mark.gpu


def _bar(nx):
    """A bar on a clamped face (every node column is held, so the iteration
    count does not depend on the length), a random start to be relaxed to 0."""
    import vpfhf_amd as V
    P = V.Problem((nx, 2, 2), (float(nx - 1), 1.0, 1.0), nu=0.3, eta=1e-5, atnum=1)
    P.set_bc([V.make_bc({4: V.ZERO})] * 3, V.make_bc())
    rng = np.random.default_rng(nx)
    P.set_fields(V=rng.uniform(0.5, 1.0, P.nn))
    return P, rng.uniform(-1e-3, 1e-3, 3 * P.nn)


# tiles: 66,669; 131,337; 262,669 (partials: 129,024 of p.q under multigrid and
# 262,144 under Jacobi, 131,072 of r.z)
@pytest.mark.parametrize("nx,pc,rtol", [(1000021, "mg", 1e-9), (1970041, "mg", 1e-9), (3940021, "jacobi", 1e-6)])
def test_u_solve_of_many_tiles(nx, pc, rtol):
    from vpfhf_amd import _lib
    pc = _lib.PC_MG if pc == "mg" else _lib.PC_JACOBI
    its = []
    for n in (3001, nx):
        P, U0 = _bar(n)
        Z = np.zeros(3 * P.nn)
        U, info = P.VF_StepU(U0, Z, rtol=rtol, pc=pc)
        assert info.status == 0
        its.append(info.iterations)
        # the recurrence's residual and the true one agree to rounding
        r, r0 = (np.linalg.norm(P.VF_UResidual(P.VecApplyDirichletBC(u, Z), Z)) for u in (U, U0))
        assert r <= 1.01 * rtol * r0, (r, r0)
        P.close()
    # the extremes of a larger sample cost a step or two; the batch lengths round it up
    assert its[1] <= 1.25 * its[0] + 4, its
