"""Long bars: grids of more workgroup tiles than the solvers keep reduction
partials for (one element in y and z, one 15-node tile per 15 nodes; the products
and the post-smoothing then reduce in a pass of their own), and axes of more than
65535 elements, whose products of two counts pass 31 bits."""
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


def _held_bar(axis, m):
    """m elements along axis, short ones, so that the coarse levels carry the
    convergence; E over three decades along it, so that they need its means."""
    import vpfhf_amd as V
    n, l = [3, 3, 3], [1.0, 1.0, 1.0]
    n[axis], l[axis] = m + 1, 0.05 * m
    P = V.Problem(tuple(n), tuple(l), nu=0.3, eta=1e-5, atnum=1)
    P.set_bc([V.make_bc({2 * ((axis + 1) % 3): V.ZERO})] * 3, V.make_bc())
    shape = [q - 1 for q in n[::-1]]
    along = np.exp(1.5 * np.log(10.0) * np.sin(2 * np.pi * (np.arange(m) + 0.5) / 1000))
    E = np.broadcast_to(along.reshape([-1 if 2 - d == axis else 1 for d in range(3)]), shape)
    P.set_fields(V=np.ones(P.nn), E_elem=np.ascontiguousarray(E).ravel())
    return P


@pytest.mark.parametrize("axis", [0, 2], ids="xz")
def test_multigrid_coefficients_of_long_axes(axis):
    """Coarse coefficients and transfers beyond 65535 elements along an axis: the
    solve takes the iterations of the same bar at half the length, a third of
    Jacobi's or fewer, and the V-cycle is positive."""
    from vpfhf_amd import _lib
    its = []
    for m in (33000, 66000):
        P = _held_bar(axis, m)
        rng = np.random.default_rng(m)
        Z, U0 = np.zeros(3 * P.nn), rng.uniform(-1e-3, 1e-3, 3 * P.nn)
        _, info = P.VF_StepU(U0, Z, rtol=1e-9, pc=_lib.PC_MG)
        assert info.status == 0
        its.append(info.iterations)
        if m == 33000:
            _, jac = P.VF_StepU(U0, Z, rtol=1e-9, pc=_lib.PC_JACOBI)
            assert 3 * info.iterations < jac.iterations, (info.iterations, jac.iterations)
        free = 1.0 - P.bc_mask("U")
        a = rng.standard_normal(3 * P.nn) * free
        assert a @ P.u_pc_apply(a) > 0.0
        P.close()
    # two samples of the same statistics: a step or two, rounded up to a batch of four
    assert abs(its[1] - its[0]) <= 4, its


def _plate(n):
    import vpfhf_amd as V
    P = V.Problem((n, n, 2), ((n - 1) / 128, (n - 1) / 128, 1 / 128), nu=0.2, atnum=2, epsilon=4 / 128, eta=1e-5,
                  alpha=0.0, beta=0.0)
    P.set_fields(V=np.ones(P.nn), VIrrev=np.ones(P.nn))
    rng = np.random.default_rng(n)
    return P, 1e-2 * rng.random(3 * P.nn), 0.5 + 0.5 * rng.random(P.nn)


def test_v_solve_of_many_chunks():
    """More chunks in the reduced system than its launches sum directly: the
    iterations of a small plate (same statistics), and the gradient asked for."""
    its = []
    for n in (201, 1001):  # 196 and 4489 chunks
        P, U, V0 = _plate(n)
        V, info = P.VF_StepV(U, V0, rtol=1e-8)
        assert info.status == 0
        its.append(info.iterations)
        P.VIJacobian_setup(U)
        g, g0 = (np.linalg.norm(P.VF_VResidual(v)) for v in (V, V0))
        assert g <= 1.01e-8 * g0, (g, g0)
        P.close()
    # a larger sample's extremes cost a step or two in each of the few Newton steps
    assert its[1] <= 1.25 * its[0] + 4, its


@pytest.mark.parametrize("n", [201, 501, 1001])
def test_v_solve_of_many_chunks_is_reproducible(n):
    """196 chunks (all resident at once), 1156 and 4489 (late workgroups start after
    the first has decided whether the CG goes on): bitwise the same every time."""
    P, U, V0 = _plate(n)
    V, info = P.VF_StepV(U, V0, rtol=1e-8)
    for _ in range(3):
        W, again = P.VF_StepV(U, V0, rtol=1e-8)
        assert again.iterations == info.iterations and np.array_equal(V, W)
    P.close()


def test_v_solve_time_follows_the_grid():
    """A CG iteration reads the coupling once, whatever the number of chunks
    (71,289 here): a few products' time each, all else included."""
    import ctypes as C
    import time
    import vpfhf_amd as vf
    from vpfhf_amd import DeviceBuffer, _lib
    P, U, V0 = _plate(4001)
    dU, dV, dy = DeviceBuffer(8 * U.size).upload(U), DeviceBuffer(8 * V0.size), DeviceBuffer(8 * V0.size)
    L, o, info = vf.load(), P.opts(rtol=1e-8), _lib.SolveInfo()

    def timed(f, n):
        t = []
        for _ in range(n):
            dV.upload(V0)
            t0 = time.perf_counter()
            vf.check(f(), P.h)
            t.append(time.perf_counter() - t0)
        return sorted(t)[n // 2]

    solve = timed(lambda: L.vfg_v_solve(P.h, dU.ptr, dV.ptr, None, C.byref(o), C.byref(info), vf.DEVICE), 3)
    product = timed(lambda: L.vfg_v_apply(P.h, dV.ptr, dy.ptr, vf.DEVICE), 9)
    # an iteration: the product and an update of three of its eight vector passes
    # (the product itself is bound by the coupling, 27 values per element)
    assert solve <= 6 * product * info.iterations, (solve, product, info.iterations)
    P.close()


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
def test_batched_multigrid_of_long_axes(mixed):
    """Members whose last level still has more than eight elements along an axis
    (the hierarchy ends at twelve levels), beside one whose last level is solved in
    one workgroup: each as alone, and as by itself outside the batch."""
    from vpfhf_amd import _lib
    from vpfhf_amd.batch import Batch
    boxes = [(0, 20000), (2, 33000), (1, 40), (0, 20000)]
    rng = np.random.default_rng(8)
    U0 = [rng.uniform(-1e-3, 1e-3, 27 * (m + 1)) for _, m in boxes]  # 3 x 3 nodes across

    def solve(pick):
        P = [_held_bar(*boxes[i]) for i in pick]
        B = Batch(P)
        Z = [np.zeros(3 * p.nn) for p in P]
        U, infos = B.u_solve([U0[i] for i in pick], Z, rtol=1e-9, mixed=mixed, pc=_lib.PC_MG)
        assert all(q.status == 0 for q in infos)
        B.close()
        single = []
        for i, p, z in zip(pick, P, Z):
            u, info = p.VF_StepU(U0[i], z, rtol=1e-9, pc=_lib.PC_MG)
            assert info.status == 0
            # both solves end within rtol of a zero load's solution, 0: their
            # residuals are what can be compared
            r0 = np.linalg.norm(p.VF_UResidual(p.VecApplyDirichletBC(U0[i], z), z))
            for v in (u, U[pick.index(i)]):
                assert np.linalg.norm(p.VF_UResidual(v, z)) <= 1.01e-9 * r0
            single.append(info.iterations)
            p.close()
        return U, [q.iterations for q in infos], single

    mix, its, single = solve([0, 1, 2, 3])
    if not mixed:  # the same algorithm; the single solve looks at its residual every few steps
        assert all(abs(a - b) <= 4 for a, b in zip(its, single)), (its, single)
    for i in range(4):
        assert np.array_equal(solve([i])[0][0], mix[i]), i
