"""The 1-D eigen-factors of the exact solves: axes with one operator share its
factors (coarse_factors), and a handle keeps the uniform level's factors until
an operator changes."""
import copy

import numpy as np
import pytest


@pytest.mark.parametrize("ndim,nc", [(2, 8), (2, 64), (3, 2), (3, 16), (3, 128)])
def test_equal_axes_share_their_factors(A, ndim, nc):
    """Every axis of a call has the factors that its operator has in a call
    where all axes differ, and they diagonalise that operator."""
    bc = np.zeros(2 * ndim, np.int32)
    bc[-2:] = 1
    dr = np.full(ndim, 1e-3)
    together = A.coarse_factors(ndim, nc, A.XYZ, np.zeros(ndim), dr, bc)
    for d in range(ndim):
        other = dr * (2.0 + np.arange(ndim))
        other[d] = dr[d]
        alone = A.coarse_factors(ndim, nc, A.XYZ, np.zeros(ndim), other, bc)
        for x, y, w in zip(together, alone, (nc * nc, nc * nc, nc)):
            assert np.array_equal(x[d * w:(d + 1) * w], y[d * w:(d + 1) * w])
        T = (np.diag(np.full(nc - 1, 1.0), 1) + np.diag(np.full(nc - 1, 1.0), -1) - 2 * np.eye(nc))
        fold = -1.0 if bc[2 * d] else 1.0
        T[0, 0] += fold
        T[-1, -1] += fold
        T *= 1e6
        n2 = nc * nc
        Vi, V = (m[d * n2:(d + 1) * n2].reshape(nc, nc) for m in together[:2])
        e = together[2][d * nc:(d + 1) * nc]
        # (128 eps of the operator's norm 4e6, over nc rounding sums)
        assert np.abs(V @ np.diag(e) @ Vi - T).max() < 128 * 2.3e-16 * 4e6 * nc
        assert np.abs(V @ Vi - np.eye(nc)).max() < 128 * 2.3e-16 * nc


@pytest.mark.gpu
@pytest.mark.parametrize("ndim,nc", [(2, 8), (3, 8), (3, 16)])
def test_kept_factors_follow_the_operator(S, A, ndim, nc):
    """A handle that has solved with another uniform level, or on another
    tree, solves as a new one does."""
    one = S.small_amr(ndim, nc=nc, uniform_lvl=3, max_lvl=4, frac=0.4, seed=3)
    one.params.mg_num_vcycles = 20
    one.params.mg_max_rel_residual = 1e-8
    wide = copy.copy(one)  # the same boxes, twice as large
    wide.extra = dict(one.extra, export=dict(one.extra["export"]))
    for k in ("dr", "r_min"):
        wide.extra["export"][k] = 2 * one.extra["export"][k]

    def solve(p, case, n):
        p.set_option(A.OPT_DIRECT_N, n)
        S.apply(p, case)
        p.put_cc(A.CC_PHI, np.zeros_like(case.ne0))  # (a solve starts from the last one's potential)
        return p.field_compute(0, False), p.get_cc(A.CC_PHI)

    def handle():
        return A.Path("gpu", ndim, nc, A.XYZ, A.PREC_MIXED)

    kept = handle()
    for case, n in ((one, 128), (one, 16), (wide, 16), (wide, 128), (one, 128)):
        new = handle()
        got, want = solve(kept, case, n), solve(new, case, n)
        new.close()
        assert got[0] == want[0]
        assert np.array_equal(got[1], want[1])
    kept.close()
