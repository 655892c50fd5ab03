"""Element forms of the batched kernels (cubic, general; coarse levels with s =
1): which one runs depends on every listed member, and on every level of its
hierarchy, so ensembles and request streams of boxes are solved in several
mixes.  Bar: a member's result is bitwise what it is alone (the forms differ by
exact factors of 1), whatever the mix, its changes and graphs on or off; alone it
agrees with the oracle within 1e-8 in FP64 and 1e-7 in the mixed form, as the
other batched solves."""
import numpy as np
import pytest

from . import scenarios as S
from .scenarios import relerr

pytestmark = pytest.mark.gpu

# nodes, lengths: cubic on every level; cubic with a general coarse level (25 x
# 17 x 9 -> 13 x 9 x 5 elements); general on every level; of one level, cubic and not
BOXES = {"cube": ((17, 17, 17), (1.0, 1.0, 1.0)),
         "odd": ((26, 18, 10), (25 / 16, 17 / 16, 9 / 16)),
         "box": ((19, 12, 9), (1.0, 2.3, 0.6)),
         "small": ((9, 8, 6), (1.0, 7 / 8, 5 / 8)),
         "smallbox": ((7, 9, 6), (1.0, 0.4, 0.9))}
MIXES = [("cube", "odd"), ("cube", "small"), ("odd", "box"), ("small", "smallbox"), ("box", "small"), tuple(BOXES)]


@pytest.fixture(scope="module")
def cases(oracle):
    out = {}
    for i, (k, (n, l)) in enumerate(BOXES.items()):
        s = S.make(n=n, l=l, seed=31 + i, nu=0.3, bcU=S.TEST1_U)
        op, F = S.to_oracle(oracle, s)
        B = oracle.vec_set_from_bc(op, "U") * 0.01
        U0 = oracle.vec_apply_dirichlet(op, np.zeros(3 * op.nn), B, "U")
        U = U0.copy()
        oracle.u_solve(op, F, U, B, rtol=1e-12)
        out[k] = (s, U0, B, U)
    return out


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
def test_batch_multigrid_forms(cases, mixed):
    from vpfhf_amd import _lib
    from vpfhf_amd.batch import Batch

    def solve(names, graph=True):
        P = [S.to_gpu(cases[k][0]) for k in names]
        B = Batch(P)
        B.set_graph(graph, 4)
        U, infos = B.u_solve([cases[k][1] for k in names], [cases[k][2] for k in names],
                             rtol=1e-10 if mixed else 1e-11, mixed=mixed, pc=_lib.PC_MG)
        assert all(i.status == 0 for i in infos)
        B.close()
        for p in P:
            p.close()
        return U

    alone = {k: solve([k])[0] for k in BOXES}
    for k, u in alone.items():
        assert relerr(u, cases[k][3]) < (1e-7 if mixed else 1e-8), (k, relerr(u, cases[k][3]))
    for mix in MIXES:
        for k, u in zip(mix, solve(mix)):
            assert np.array_equal(u, alone[k]), (mix, k)
    for k, u in zip(BOXES, solve(list(BOXES), graph=False)):
        assert np.array_equal(u, alone[k]), k


@pytest.mark.parametrize("n,l", [((18, 10, 12), (17 / 8, 9 / 8, 11 / 8)), ((11, 12, 9), (1.0, 2.3, 0.6))],
                         ids=["cubic", "general"])
@pytest.mark.parametrize("with_box", [False, True], ids=["one", "mix"])
def test_batch_fp32_apply_forms(oracle, n, l, with_box):
    # FP32 rounds its inputs too: 1e-5 as for the other FP32 applies
    from vpfhf_amd.batch import Batch
    sc = [S.make(n=n, l=l, seed=3, nu=0.3)]
    if with_box:
        sc.append(S.make(n=(9, 17, 10), l=(0.7, 1.0, 2.0), seed=4, nu=0.3))
    P = [S.to_gpu(s) for s in sc]
    B = Batch(P)
    for s, y in zip(sc, B.u_apply([s["x"] for s in sc], fp32=True)):
        op, F = S.to_oracle(oracle, s)
        ref = oracle.u_jacobian(op, F) @ s["x"]
        assert np.abs(y - ref).max() <= 1e-5 * np.abs(ref).max()
    B.close()
    for p in P:
        p.close()


class _Stream:
    """Requests of box-shaped problems (serve.RequestSet builds cubes)."""

    def __init__(self, items):  # (nodes, lengths, seed, iterations)
        from vpfhf_amd.host import Request
        self.arr = (Request * len(items))()
        self.keep, self.U, self.V, self.text, self.fields = [], [], [], [], []
        for r, (n, l, seed, am) in zip(self.arr, items):
            rng = np.random.default_rng(seed)
            nn, ne = int(np.prod(n)), int(np.prod([m - 1 for m in n]))
            h = l[0] / (n[0] - 1)
            from vpfhf_amd import workloads
            text = "-n %d,%d,%d -l %r,%r,%r\n" % (n + l)
            text += "-E 1.0 -nu 0.25 -beta 0.0 -alpha 1e-5 -Gc 1.0 -epsilon %r -eta 1e-5 -atnum 1\n" % (2 * h)
            text += "-U_ksp_rtol 1e-10 -npc 1 -pressurize -altmintol 0.0\n"
            text += "-pc0_center %r,%r,%r -pc0_r %r -pc0_theta 20. -pc0_phi 30. -pc0_thickness %r\n" % (
                l[0] / 2, l[1] / 2, l[2] / 2, 0.3 * min(l), 3 * h)
            text += workloads.CLAMPED_OPTIONS
            f = dict(E_elem=np.exp(0.4 * rng.standard_normal(ne)), theta=np.zeros(nn), thetaRef=np.zeros(nn),
                     pressure=np.full(nn, 2e-3))
            U, V = np.zeros(3 * nn), np.zeros(nn)
            opt = text.encode()
            r.options = opt
            r.E_elem, r.theta, r.thetaRef, r.pressure = [f[k].ctypes.data for k in
                                                         ("E_elem", "theta", "thetaRef", "pressure")]
            r.am_maxit = am
            r.U_out, r.V_out = U.ctypes.data, V.ctypes.data
            self.keep.append((opt, f))
            self.U.append(U)
            self.V.append(V)
            self.text.append(text)
            self.fields.append(f)

    def __len__(self):
        return len(self.arr)


# a general request joins cubes and leaves before they finish, a cube with a
# general coarse level takes its place, and the engine ends with cubes only
STREAM = [((13, 13, 13), (1.0, 1.0, 1.0), 1, 6), ((14, 11, 9), (1.0, 2.0, 0.5), 2, 1),
          ((11, 11, 11), (1.0, 1.0, 1.0), 3, 1), ((26, 18, 10), (25 / 16, 17 / 16, 9 / 16), 4, 1),
          ((12, 12, 12), (1.0, 1.0, 1.0), 5, 2), ((7, 9, 6), (1.0, 0.4, 0.9), 6, 1),
          ((15, 15, 15), (1.0, 1.0, 1.0), 7, 2)]


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
def test_engine_form_changes(mixed):
    from vpfhf_amd import serve
    from vpfhf_amd.host import Host, options
    R = _Stream(STREAM)
    res, st = serve.serve(R, max_slots=3, realtime=False, mixed=mixed)
    assert all(r["status"] == 0 for r in res) and st["max_resident"] == 3
    for i, item in enumerate(STREAM):
        A = _Stream([item])
        ra, _ = serve.serve(A, max_slots=1, realtime=False, mixed=mixed)
        assert ra[0]["status"] == 0 and ra[0]["u_its"] == res[i]["u_its"] and ra[0]["v_its"] == res[i]["v_its"], i
        assert np.array_equal(A.U[0], R.U[i]) and np.array_equal(A.V[0], R.V[i]), i
        H = Host(options(R.text[i]))
        H.set_inputs(**R.fields[i])
        H.fields_initialize()
        H.set_bcu(1.0)
        H.timestep_prepare()
        info = H.altmin(maxit=item[3])
        U, V, _ = H.state()
        H.close()
        assert info.status == 0 and info.iterations == res[i]["am_iterations"]
        # u to 1e-10 of its residual and V to 1e-8 of its gradient in each iteration
        assert relerr(R.U[i], U) < 1e-6 and relerr(R.V[i], V) < 1e-6, (i, relerr(R.U[i], U), relerr(R.V[i], V))
