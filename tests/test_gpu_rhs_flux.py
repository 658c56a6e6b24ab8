"""The ghost fill and coarse rhs in one launch (k_gc_rhs, smaller 2D levels)
against the two launches of large levels: the same bits."""
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
