"""The FP32 half-sweeps of one row per lane (k_gsrb_split2d on large levels of
8^2 boxes, k_gsrb_row3d on 8^3 boxes) against the box-staging half-sweep
(AFGPU_OPT_BOX_LDS): the same bits, with refinement boundaries, both
coordinate systems, box counts that fill no workgroup, and masked runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _both(A, make, drive, ivs):
    out = []
    for box_lds in (0, 1):
        p = make()
        p.set_option(A.OPT_BOX_LDS, box_lds)
        infos = drive(p)
        out.append((infos, [p.get_cc(iv) for iv in ivs]))
        p.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        assert np.array_equal(a, b)


def _tight(case, photoi=False):
    case.params.mg_num_vcycles = 20
    case.params.mg_max_rel_residual = 1e-8
    case.params.photoi_enabled = int(photoi)
    return case


@pytest.mark.parametrize("uniform,top,frac,seed", [(1, 3, 0.9, 3), (2, 4, 0.4, 5), (3, 4, 0.1, 9), (3, 5, 0.3, 7)])
def test_rows_of_3d_boxes(S, A, uniform, top, frac, seed):
    case = _tight(S.small_amr(3, nc=8, uniform_lvl=uniform, max_lvl=top, frac=frac, seed=seed), photoi=True)
    _both(A, lambda: S.apply(A.Path("gpu", 3, 8, A.XYZ, A.PREC_MIXED), case),
          lambda p: [p.field_compute(0, False)] + [p.step() for _ in range(2)],
          (A.CC_PHI, A.CC_ELECTRON, A.CC_PHOTO))


@pytest.mark.parametrize("coord", ["CYL", "XYZ"])
def test_rows_of_large_2d_levels(S, A, coord):
    coord = getattr(A, coord)
    case = _tight(S.small_amr(2, coord=coord, uniform_lvl=7, max_lvl=9, frac=0.5, seed=17))
    t = case.extra["export"]
    assert np.bincount(t["lvl"])[8:].min() >= 7168
    _both(A, lambda: S.apply(A.Path("gpu", 2, 8, coord, A.PREC_MIXED), case),
          lambda p: [p.field_compute(0, False), p.step()], (A.CC_PHI, A.CC_ELECTRON))


def test_rows_of_large_2d_forest(S, A):
    ens = S.ensemble(level_list=[8, 5, 7, 8], num_vcycles=20, rel_residual=1e-8)
    _both(A, lambda: S.apply_ensemble(A.Path("gpu", 2, 8, A.CYL, A.PREC_MIXED), ens),
          lambda p: [[list(x) for x in p.field_compute_runs(0, have_guess=False)], p.step_ensemble()],
          (A.CC_PHI, A.CC_ELECTRON))
