"""The ghost fill and coarse rhs in one launch (k_gc_rhs, smaller 2D levels)
against the two launches of large levels, the two forms of the residual
restriction of FP32 16^3 boxes, and k_flux's two homes of the transport table:
the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
def test_copies_of_a_run_in_small_and_large_forests(S, A, mixed):
    """A run's solution does not depend on how many copies of it the forest
    holds: 2, and 447 and 449, with 16 boxes on its level 3 on either side of
    the line between one launch and two (7168 boxes)."""
    one = S.small_amr(2, coord=A.CYL, uniform_lvl=3, max_lvl=5, frac=0.5, seed=29)
    one.params.mg_num_vcycles = 12
    one.params.mg_max_rel_residual = 1e-8
    n1 = one.extra["export"]["n_boxes"]

    def solve(n):
        t, ne0, offs = S.merge_forest([one] * n)
        p = A.Path("gpu", 2, 8, A.CYL, A.PREC_MIXED if mixed else A.PREC_FP64)
        S.apply_ensemble(p, S.Ensemble([one] * n, t, ne0, offs, np.full(n, one.voltage), name="copies"))
        info = [list(x) for x in p.field_compute_runs(0, have_guess=False)]
        phi = p.get_cc(A.CC_PHI).reshape(n, -1)
        p.close()
        return info, phi

    info, want = solve(2)
    assert np.array_equal(want[0], want[1]) and n1 > 21
    for n in (447, 449):
        got = solve(n)
        for a, b in zip(got[0], info):
            assert list(a) == [b[0]] * n
        assert np.array_equal(got[1], np.broadcast_to(want[0], got[1].shape))


def test_restriction_of_small_and_large_3d_levels(S, A):
    """FP32 levels of 16^3 boxes are restricted a cell per thread up to one
    box per CU and a parent cell per thread above: 2, 10 and 11 copies of a
    run with 24 boxes and refinement boundaries on level 3 lie on either side
    of that line (256 boxes)."""
    one = S.small_amr(3, nc=16, uniform_lvl=2, max_lvl=3, frac=0.4, seed=37)
    one.params.mg_num_vcycles = 12
    one.params.mg_max_rel_residual = 1e-8
    assert list(np.bincount(one.extra["export"]["lvl"])) == [0, 1, 8, 24]
    out = []
    for n in (2, 10, 11):
        t, ne0, offs = S.merge_forest([one] * n)
        p = A.Path("gpu", 3, 16, A.XYZ, A.PREC_MIXED)
        S.apply_ensemble(p, S.Ensemble([one] * n, t, ne0, offs, np.full(n, one.voltage), name="copies"))
        info = [list(x) for x in p.field_compute_runs(0, have_guess=False)]
        out.append((info, p.get_cc(A.CC_PHI).reshape(n, -1)))
        p.close()
    want = out[0][1][0]
    for info, phi in out:
        for a, b in zip(info, out[0][0]):
            assert list(a) == [b[0]] * len(phi)
        assert np.array_equal(phi, np.broadcast_to(want, phi.shape))


@pytest.mark.parametrize("ndim,nc", [(2, 8), (2, 16), (3, 8), (3, 16)])
def test_flux_with_the_table_in_lds_and_in_memory(S, A, ndim, nc):
    """A transport table of more rows than LDS holds, its first rows the
    small one's and its others never reached, gives the same step."""
    case = S.small_amr(ndim, nc=nc, uniform_lvl=2, max_lvl=3, frac=0.5, seed=31)
    out = []
    for rows in (case.tdata["n"], 1024, 1025):
        tb = dict(case.tdata)
        for k in ("td", "chem"):
            cols = np.asarray(tb[k]).reshape(-1, tb["n"])
            tb[k] = np.ascontiguousarray(np.concatenate([cols, np.repeat(cols[:, -1:], rows - tb["n"], 1)], 1))
        tb["n"] = rows
        p = A.Path("gpu", ndim, nc, A.XYZ, A.PREC_MIXED)
        S.apply(p, case)
        p.set_tables(tb)
        out.append([p.field_compute(0, False)] + [p.step() for _ in range(2)] + [p.get_cc(A.CC_ELECTRON)])
        p.close()
    for o in out[1:]:
        assert o[:-1] == out[0][:-1]
        assert np.array_equal(o[-1], out[0][-1])
