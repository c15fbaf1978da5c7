"""Explicit Schur solve at the sizes where its blocked Cholesky changes shape:
orders of S (9 per camera) around the 16-column tiles and the 64-column blocks,
and whole blocks only.  One LM iteration from the
generator's start against the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Cameras: n = 18 (16 + 2), 63, 72 (64 + 8), 81 (64 + 16 + 1), 126, 135
# (128 + 7), 144 (whole tiles), 198, 261, 576 (whole blocks).
CAMS = [2, 7, 8, 9, 14, 15, 16, 22, 29, 64]


@pytest.mark.parametrize("ncam", CAMS)
def test_one_explicit_iteration_is_the_oracles(mba, O, ncam):
    npt = 30 * ncam
    tmax = min(ncam, 6)
    d = O.generate(O.make_spec(num_cameras=ncam, num_points=npt, track_min=2, track_max=tmax, seed=ncam))
    so, _ = O.solve(O.Scene(d), O.default_options(linear_solver=0, max_num_iterations=1))
    # FP64: the step's error is a few n eps cond, with cond <= ~1e8 under the
    # first damping: 1e-6 of the step, and the cost's change is of second order
    # in what the damping leaves free.  FP32 S, refined against itself: its
    # entries carry 6e-8, so the directions the cost depends on (cond <= ~1e4)
    # are good to 6e-4.
    for precision, tol in ((mba.PRECISION_FP64, 1e-8), (mba.PRECISION_MIXED, 1e-3)):
        print(f"cameras {ncam} precision {precision}", flush=True)
        p = mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"])
        s = mba.solve(p, mba.default_options(linear_solver=mba.EXPLICIT_SCHUR, precision=precision,
                                             max_num_iterations=1))
        assert [it.step_is_successful for it in s.iterations][1:] == [1]
        assert np.all(np.isfinite(p.cameras)) and np.all(np.isfinite(p.points))
        np.testing.assert_allclose(s.initial_cost, so.initial_cost, rtol=1e-6)
        np.testing.assert_allclose(s.final_cost, so.final_cost, rtol=tol, atol=1e-9 * so.initial_cost)
