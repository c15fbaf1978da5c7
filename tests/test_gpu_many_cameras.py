"""Point-major kernels of a single large problem with more cameras than the LDS
records hold (cooperative camera reads) against the general path: the same
problem with more rows per lane is below the launch size from which the
cooperative reads are taken.  Both sum the same rows' terms in different
orders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(O):
    # 140,000 points with 2..19 rows: 4 rows a lane give > 1,024 workgroups of
    # 256 threads, 64 rows a lane give 547; waves end with 0..63 rows left.
    return O.generate(O.make_spec(num_cameras=2300, num_points=140001, track_min=2, track_max=19, outlier_frac=0.05,
                                  seed=12))


@pytest.mark.parametrize("huber", [0.0, 4.0])
@pytest.mark.parametrize("precision", [0, 1])
def test_cooperative_reads_give_the_general_paths_blocks(mba, scene, precision, huber):
    d = scene
    x = np.random.default_rng(5).standard_normal(9 * 2300)
    got = []
    for rpl in (4, 64):
        print(f"precision {precision} huber {huber} rows per lane {rpl}", flush=True)
        p = mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"])
        o = mba.default_options(precision=precision, linear_solver=mba.IMPLICIT_SCHUR_PCG, huber_a=huber,
                                point_rows_per_lane=rpl)
        with mba.Context(p, o) as c:
            cost = c.lm_pass(1e4)
            got.append(dict(c.read_schur(), y=np.array(c.schur_matvec(x)), cost=np.array([cost])))
    a, b = got
    # Blocks and gradients: sums of up to ~700 terms, 700 eps of the largest.
    # rhs and y = S x add V^-1 applied to a point's sums (~20 terms, 20 eps),
    # amplified by at most the damped blocks' condition (~1e4) at single points
    # and averaged over a camera's ~700: 1e4 20 eps / sqrt(700).
    eps = 2.3e-16 if precision == 0 else 6e-8
    for k in a:
        tol = (1e4 * 20 / 26 if k in ("rhs", "y") else 700) * eps
        err = np.max(np.abs(a[k] - b[k])) / np.max(np.abs(b[k]))
        print(f"  {k}: {err:.1e} (<= {tol:.1e})", flush=True)
        assert err <= tol, k
