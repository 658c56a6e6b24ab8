"""The uniform-level solve of the mixed form's inner cycle: the whole-line
transforms on the matrix cores (k_lc_x, k_lc_line; the last axis in place)
against the vector transforms (AFGPU_OPT_DIRECT_MFMA 0), after one inner cycle
and after whole solves, at every size they exist for.

Tolerance: both transform in FP64 and differ by about 1e-13 of the solution's
maximum, so an FP32 value of the solved level changes by one unit in the last
place at most, 2^-23 of that maximum; each half-sweep and prolongation above
(at most 9 on the one or two finer levels here) adds no more than another.
16 units: 2e-6.  The charges are random in every cell, so every mode takes
part: without the highest mode of one axis the solution changes by 1.6e-3 of
its maximum or more at all of these sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 16 * 2.0 ** -23


def _handle(A, D, nc, coord, mfma, fold=1):
    p = A.Path("gpu", D, nc, coord, A.PREC_MIXED)
    p.set_option(A.OPT_DIRECT_MFMA, mfma)
    p.set_option(A.OPT_DIRECT_FOLD, fold)
    return p


def _charges(A, p, ne0, seed):
    p.put_cc(A.CC_POS_ION, ne0 + np.random.default_rng(seed).uniform(-1e17, 1e17, ne0.shape))


def _close(a, b):
    assert np.abs(a).max() > 0
    assert np.abs(a - b).max() <= TOL * np.abs(b).max()


# (boxes of nc cells, uniform level: nc 2^(level - 1) cells per axis; finest level)
@pytest.mark.parametrize("nc,uniform,top", [(8, 3, 3), (8, 3, 5), (16, 2, 2), (16, 2, 3), (8, 4, 4), (16, 3, 4),
                                            (16, 4, 4), (16, 4, 5), (8, 5, 5)])
def test_one_inner_cycle_3d(S, A, nc, uniform, top):
    case = S.small_amr(3, nc=nc, uniform_lvl=uniform, max_lvl=top, frac=0.1, seed=41)
    case.params.mg_num_vcycles = 1
    got = []
    for mfma, fold in ((0, 1), (1, 1), (1, 0)):
        p = S.apply(_handle(A, 3, nc, A.XYZ, mfma, fold), case)
        _charges(A, p, case.ne0, 1)
        assert p.field_compute(0, have_guess=True)[0] == 1
        got.append(p.get_cc(A.CC_PHI))
        p.close()
    for g in got[1:]:
        _close(g, got[0])


@pytest.mark.parametrize("coord", ["XYZ", "CYL"])
@pytest.mark.parametrize("nc,levels", [(8, (3, 5, 4)), (16, (2, 4, 3)), (8, (4, 6, 5)), (16, (3, 4, 5)), (8, (5, 6, 7)),
                                       (16, (4, 6, 5)), (8, (5,)), (16, (3,))])
def test_forests_with_runs_masked(S, A, coord, nc, levels):
    """Runs of different depths, each masked out when it has converged: one
    cycle from zero, the solve from there, and one for other charges, which
    starts from what the cycles without the masked runs left."""
    coord = getattr(A, coord)
    cases = [S.make_case(2, nc, coord, [4e-3, 4e-3], 1e4 + 500.0 * r, lvl, [0.0, 2.8e-3], rng_seed=50 + r)
             for r, lvl in enumerate(levels)]
    t, ne0, offs = S.merge_forest(cases)
    ens = S.Ensemble(cases, t, ne0, offs, np.array([c.voltage for c in cases]), name="direct")
    params = cases[0].params
    params.mg_max_rel_residual = 1e-8
    got = []
    for mfma in (0, 1):
        p = S.apply_ensemble(_handle(A, 2, nc, coord, mfma), ens)
        p.set_voltage(ens.voltages[0])  # (of a single run)
        n, phi = [], []
        for seed, cycles in ((1, 1), (1, 30), (2, 30)):
            params.mg_num_vcycles = cycles
            p.set_params(params)
            _charges(A, p, ne0, seed)
            n.append(p.field_compute_runs(0, have_guess=True)[0])
            phi.append(p.get_cc(A.CC_PHI))
        got.append((np.array(n), phi))
        p.close()
    assert np.abs(got[0][0] - got[1][0]).max() <= 1
    for a, b in zip(got[1][1], got[0][1]):
        _close(a, b)
