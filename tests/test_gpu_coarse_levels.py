"""The coarse levels of the FP64 cycles in one workgroup per run (k_tail)
against the level kernels, which run instead while launches are timed: every
cell of every box equal bit for bit, at the box sizes, coordinate systems and
numbers of levels where the levels held end differently."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cases(S, A):
    for coord in (A.XYZ, A.CYL):
        for lvl in (1, 2, 4, 5):
            yield S.make_case(2, 8, coord, [4e-3, 4e-3], 1e4, lvl, [0.0, 2.8e-3])
        yield S.small_amr(2, nc=16, coord=coord, uniform_lvl=3, max_lvl=5)
        yield S.small_amr(2, nc=8, coord=coord, uniform_lvl=2, max_lvl=5)
    for nc in (8, 16):
        yield S.small_amr(3, nc=nc, uniform_lvl=2, max_lvl=3 if nc == 16 else 4)
        yield S.make_case(3, nc, A.XYZ, [4e-3] * 3, 1e4, 1, [2e-3, 2e-3, 2.8e-3])


@pytest.mark.parametrize("n", range(16))
def test_one_workgroup_equals_level_kernels(S, A, n):
    case = list(_cases(S, A))[n]
    got = []
    for timed in (0, 1):
        p = S.apply(A.Path("gpu", case.D, case.nc, case.coord), case)
        p.lib.afgpu_kernel_timing(p.h, timed)
        for _ in range(2):  # (the second pass replays the captured graphs)
            p.mg_fas_fmg(A.OP_POISSON, True, False)
            p.mg_fas_vcycle(A.OP_POISSON, True)
            p.mg_fas_fmg(A.OP_POISSON, True, True)
        res = p.tree_maxabs_cc(A.CC_TMP)
        n_cyc = p.field_compute(0, have_guess=True)
        got.append([p.get_cc(iv) for iv in (A.CC_PHI, A.CC_RHS, A.CC_TMP)] + [np.array([res, *n_cyc])])
        p.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_forest_with_runs_masked(S, A):
    """Runs of different depths: masked runs are left as they are."""
    ens = S.ensemble(level_list=[2, 5, 3, 4], num_vcycles=30, rel_residual=1e-7)
    got = []
    for timed in (0, 1):
        p = S.apply_ensemble(A.Path("gpu", 2, 8, A.CYL, A.PREC_FP64), ens)
        p.lib.afgpu_kernel_timing(p.h, timed)
        n, r = p.field_compute_runs(0, have_guess=False)
        infos = p.step_ensemble()
        got.append([p.get_cc(iv) for iv in (A.CC_PHI, A.CC_RHS, A.CC_TMP, A.CC_ELECTRON)] +
                   [n, r, np.array([i["n_vcycles"] for i in infos])])
        p.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
