"""u-apply in moment form against the assembled oracle operator: grids whose
last tile owns one node or all of them (7-, 15-node tiles), grids on both sides
of the FP32 tile switch, cubic and non-cubic elements."""
import numpy as np
import pytest

from . import scenarios as S

pytestmark = pytest.mark.gpu

GRIDS = [(8, 8, 3), (15, 9, 4), (22, 15, 5), (23, 16, 2), (61, 30, 3), (64, 8, 6), (65, 8, 3), (30, 61, 2)]


@pytest.mark.parametrize("cubic", [True, False], ids=["cubic", "stretched"])
@pytest.mark.parametrize("n", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_u_apply_moment_form(oracle, n, cubic):
    # an entry sums about 900 products of both signs: 900 eps = 2e-13 (FP64)
    # at worst; FP32 rounds its inputs too, 1e-5 as for the other FP32 applies
    l = tuple((m - 1) / 8.0 for m in n) if cubic else (1.0, 2.3, 0.6)
    s = S.make(n=n, l=l, seed=3 * sum(n), nu=0.3, bcU=S.MIXED_U)
    op, F = S.to_oracle(oracle, s)
    P = S.to_gpu(s)
    ref = oracle.u_jacobian(op, F) @ s["x"]
    scale = np.abs(ref).max()
    assert np.abs(P.UIJacobian_mult(s["x"]) - ref).max() <= 1e-12 * scale
    assert np.abs(P.UIJacobian_mult(s["x"], fp32=True) - ref).max() <= 1e-5 * scale
    P.close()


@pytest.mark.parametrize("n", [(66, 60, 58), (65, 97, 81), (9, 40, 23)], ids=["non-nested", "nested", "flat"])
def test_vcycle_transfers(n):
    """The V-cycle is symmetric only if restriction and prolongation are each
    other's transpose and every level's operator is symmetric: one entry per
    thread (more than 2^16 coarse entries), four lanes per entry, directions
    that are not coarsened."""
    s = S.make(n=n, seed=sum(n), nu=0.3, bcU=S.MIXED_U)
    P = S.to_gpu(s)
    free = 1.0 - P.bc_mask("U")
    rng = np.random.default_rng(n[0])
    a, b = (rng.standard_normal(3 * P.nn) * free for _ in range(2))
    Ma, Mb = P.u_pc_apply(a), P.u_pc_apply(b)
    # FP32 throughout: 1e-5 of the norms, as for one FP32 apply
    assert abs(a @ Mb - b @ Ma) <= 1e-5 * np.linalg.norm(a) * np.linalg.norm(Mb)
    assert a @ Ma > 0.0
    P.close()


def test_vcycle_long_column():
    """More node planes than a launch has block rows (65535)."""
    s = S.make(n=(3, 2, 66001), l=(1.0, 0.5, 33000.0), seed=7, bcU=S.MIXED_U)
    P = S.to_gpu(s)
    free = 1.0 - P.bc_mask("U")
    rng = np.random.default_rng(7)
    a, b = (rng.standard_normal(3 * P.nn) * free for _ in range(2))
    Ma, Mb = P.u_pc_apply(a), P.u_pc_apply(b)
    # FP32 throughout: 1e-5 of the norms, as for one FP32 apply
    assert abs(a @ Mb - b @ Ma) <= 1e-5 * (np.linalg.norm(a) * np.linalg.norm(Mb) + np.linalg.norm(b) * np.linalg.norm(Ma))
    P.close()


@pytest.mark.parametrize("unilateral", [0, 1], ids=["linear", "nocompression"])
@pytest.mark.parametrize("n", [(2, 2, 2), (17, 18, 3), (18, 33, 20), (115, 114, 10), (18, 18, 1101)], ids=lambda n: "x".join(map(str, n)))
def test_energies_modal_form(oracle, n, unilateral):
    """Element tiles that are full, have one element or end in a ragged layer
    group, on both sides of the layer-group switch; AT1 and AT2."""
    # per-cell sums of 27 terms of order one operation each, 1e-12 as for the
    # other diagnostics; signed totals against the sum of their magnitudes
    for atnum in (1, 2):
        s = S.make(n=n, l=(1.0, 2.3, 0.6), seed=sum(n) + atnum, nu=0.3, atnum=atnum, unilateral=unilateral)
        s["theta"] = s["theta"] + 50.0
        op, F = S.to_oracle(oracle, s)
        P = S.to_gpu(s)
        ref = oracle.energy_fields(op, F, s["U"], s["V"])
        ef = P.energy_fields(s["U"], s["V"])
        for c in range(3):
            assert np.abs(ef[:, c] - ref[:, c]).max() <= 1e-12 * np.abs(ref[:, c]).max(), c
        el, _, pw, se = P.energies(s["U"], s["V"])
        for got, r in zip((el, pw, se), ref.T):
            assert abs(got - r.sum()) <= 1e-12 * np.abs(r).sum()
        vol, cf = P.VolumetricCrackOpening(s["U"], s["V"], cellfield=True)
        rvol, rcf = oracle.crack_volume(op, s["U"], s["V"], cellfield=True)
        assert np.abs(cf - rcf).max() <= 1e-12 * np.abs(rcf).max()
        assert abs(vol - rvol) <= 1e-12 * np.abs(rcf).mean() * np.prod(s["l"])
        P.close()


@pytest.mark.parametrize("pressurize", [True, False], ids=["pressure", "dry"])
@pytest.mark.parametrize("n", [(2, 2, 2), (15, 9, 4), (16, 31, 3), (23, 16, 5), (61, 30, 3)], ids=lambda n: "x".join(map(str, n)))
def test_u_loads_moment_form(oracle, n, pressurize):
    # b sums 8 elements of some 30 terms each, the residual about 900 products
    # more: 900 eps = 2e-13, 1e-12 as for the other operators
    s = S.make(n=n, l=(1.0, 2.3, 0.6), seed=5 * sum(n), nu=0.3, bcU=S.MIXED_U, pressurize=pressurize, alpha=1e-3)
    op, F = S.to_oracle(oracle, s)
    P = S.to_gpu(s)
    b, ref = P.u_rhs(), oracle.u_rhs(op, F)
    assert np.abs(b - ref).max() <= 1e-12 * np.abs(ref).max()
    U, BCU = s["U"], 0.3 * s["x"]
    r, rref = P.VF_UResidual(U, BCU), oracle.u_residual(op, F, U, BCU)
    assert np.abs(r - rref).max() <= 1e-12 * np.abs(rref).max()
    P.close()


@pytest.mark.parametrize("unilateral", [0, 1], ids=["linear", "nocompression"])
@pytest.mark.parametrize("n", [(2, 2, 2), (15, 16, 4), (31, 9, 5), (46, 17, 3)], ids=lambda n: "x".join(map(str, n)))
def test_v_setup_moment_form(oracle, n, unilateral):
    # energies of 27 points with mixed-sign strains, then 8 x 8 products per
    # row entry: 1e-12 as for the other operators
    for atnum in (1, 2):
        s = S.make(n=n, l=(1.0, 2.3, 0.6), seed=7 * sum(n) + atnum, nu=0.3, atnum=atnum, unilateral=unilateral,
                   bcV=S.MIXED_V)
        op, F = S.to_oracle(oracle, s)
        P = S.to_gpu(s)
        P.VIJacobian_setup(s["U"])
        b, rb = P.v_rhs(), oracle.v_rhs(op, F, s["U"])
        assert np.abs(b - rb).max() <= 1e-12 * np.abs(rb).max()
        y, ry = P.VIJacobian_mult(s["xv"]), oracle.v_jacobian(op, F, s["U"]) @ s["xv"]
        assert np.abs(y - ry).max() <= 1e-12 * np.abs(ry).max()
        P.close()


def test_batch_forms(oracle):
    """Members with equal spacings, and mixed with one without: the batched
    solves give each member what it gives alone, in either form."""
    from vpfhf_amd.batch import Batch
    boxes = [((9, 9, 9), (1.0, 1.0, 1.0)), ((18, 10, 12), (17 / 8, 9 / 8, 11 / 8)), ((11, 12, 9), (1.0, 2.3, 0.6))]
    sc = [S.make(n=n, l=l, seed=i, nu=0.3) for i, (n, l) in enumerate(boxes)]
    alone = {}
    for pick in ([0], [1], [2], [0, 1], [0, 1, 2]):
        P = [S.to_gpu(sc[i]) for i in pick]
        B = Batch(P)
        y = B.u_apply([sc[i]["x"] for i in pick])
        for i, yi in zip(pick, y):
            op, F = S.to_oracle(oracle, sc[i])
            ref = oracle.u_jacobian(op, F) @ sc[i]["x"]
            # one apply: 1e-12 as above; the forms differ by exact factors of 1 only
            assert np.abs(yi - ref).max() <= 1e-12 * np.abs(ref).max()
            if len(pick) == 1:
                alone[i] = yi
            else:
                assert np.array_equal(yi, alone[i])
        B.close()
        for p in P:
            p.close()


@pytest.mark.parametrize("n", [(2, 2, 2), (8, 15, 4), (9, 16, 31), (46, 17, 3), (47, 46, 30)], ids=lambda n: "x".join(map(str, n)))
def test_u_diag_moment_form(oracle, n):
    # 8 elements of some 30 positive terms each: 240 eps = 5e-14, 1e-12 as for
    # the other operators, entry by entry
    s = S.make(n=n, l=(1.0, 2.3, 0.6), seed=3 * sum(n), nu=0.3, bcU=S.MIXED_U)
    op, F = S.to_oracle(oracle, s)
    P = S.to_gpu(s)
    ref = oracle.u_jacobian(op, F).diagonal()
    assert np.all(np.abs(P.u_diag() - ref) <= 1e-12 * np.abs(ref))
    P.close()
