"""The device-built layout and pair list against the host-built layout: the
same problem through both (MBA_DEVICE_LAYOUT_MIN at context creation) must give
the same values bit for bit, since the two put points, rows and camera-major
rows in the same order and every sum runs in that order.  Structures on which
an ordering can go wrong: observations in shuffled order, repeated
observations, constant cameras, points and cameras without observations, a
window without observations, tracks around the sort's tile and the walk's
limits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(O, ncam, npt, tmax, seed):
    d = O.generate(O.make_spec(num_cameras=ncam, num_points=npt, track_min=2, track_max=tmax, outlier_frac=0.05,
                               seed=seed))
    return {k: np.array(v) for k, v in d.items() if k in ("cam_init", "pt_init", "obs", "cam_idx", "pt_idx")}


def _variant(O, name):
    """(scene, camera_constant)"""
    rng = np.random.default_rng(3)
    d = _scene(O, 20, 1500, 6, 5)
    const = None
    if name == "shuffled":
        o = rng.permutation(len(d["obs"]))
        d.update(obs=d["obs"][o], cam_idx=d["cam_idx"][o], pt_idx=d["pt_idx"][o])
    elif name == "repeated":
        o = np.sort(np.concatenate([np.arange(len(d["obs"])), rng.integers(0, len(d["obs"]), 300)]))
        d.update(obs=d["obs"][o], cam_idx=d["cam_idx"][o], pt_idx=d["pt_idx"][o])
    elif name == "constant":
        const = np.zeros(20, np.uint8)
        const[[0, 7, 19]] = 1
    elif name == "unobserved":
        # Points 0, 40.. and 1499 and one more camera are never observed.
        keep = ~np.isin(d["pt_idx"], [0, 40, 41, 42, 1499])
        d.update(obs=d["obs"][keep], cam_idx=d["cam_idx"][keep], pt_idx=d["pt_idx"][keep],
                 cam_init=np.vstack([d["cam_init"], d["cam_init"][:1]]))
    elif name == "long_tracks":
        d = _scene(O, 150, 4200, 150, 9)
    return d, const


def _problem(mba, d, const):
    return mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"], const)


@pytest.mark.parametrize("name", ["plain", "shuffled", "repeated", "constant", "unobserved", "long_tracks"])
@pytest.mark.parametrize("precision,solver", [(0, 0), (1, 1)])
def test_device_layout_is_the_host_layout(mba, O, monkeypatch, name, precision, solver):
    d, const = _variant(O, name)
    got = []
    for least in ("1", "1000000000"):
        print(f"layout: {name} precision {precision} solver {solver} least rows {least}", flush=True)
        monkeypatch.setenv("MBA_DEVICE_LAYOUT_MIN", least)
        o = mba.default_options(precision=precision, linear_solver=solver, huber_a=4.0, max_num_iterations=3)
        p = _problem(mba, d, const)
        with mba.Context(p, o) as c:
            cost = c.lm_pass(1e4)
            b = c.read_schur()
            scale = c.read_scale()
        s = mba.solve(p, o)
        got.append([np.array(cost), *[b[k] for k in sorted(b)], *scale, p.cameras, p.points, np.array(s.final_cost)])
    for x, y in zip(*got):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("solver", [0, 1])
def test_device_layout_of_a_batch(mba, O, monkeypatch, solver):
    scenes = [_scene(O, 5 + 7 * k, 90 + 200 * k, 4 + k, 20 + k) for k in range(4)]
    empty = dict(scenes[0], obs=np.zeros((0, 2)), cam_idx=np.zeros(0, np.int32), pt_idx=np.zeros(0, np.int32))
    # A batch's windows sum their costs with atomics in either layout, so from
    # the second iteration on a radius may differ in its last bits.  Explicit
    # steps follow it to 1e-9.  A PCG solve may then stop an iteration apart
    # (the same layout run twice does), so it takes one iteration, which no
    # atomic sum reaches: bit for bit.
    iterations, atol = ((3, 1e-9), (1, 0.0))[solver]
    got = []
    for least in ("1", "1000000000"):
        print(f"layout: batch solver {solver} least rows {least}", flush=True)
        monkeypatch.setenv("MBA_DEVICE_LAYOUT_MIN", least)
        probs = [_problem(mba, d, None) for d in (scenes[0], empty, *scenes[1:])]
        sums = mba.solve_batched(probs, mba.default_options(linear_solver=solver, max_num_iterations=iterations,
                                                             eta=1e-6))
        got.append(([(s.num_e_blocks, s.num_f_blocks, s.termination_type) for s in sums],
                    np.concatenate([p.cameras for p in probs]), np.concatenate([p.points for p in probs])))
    assert got[0][0] == got[1][0]
    for x, y in zip(got[0][1:], got[1][1:]):
        np.testing.assert_allclose(x, y, rtol=0, atol=atol)


@pytest.mark.parametrize("solver", [0, 1])
def test_device_layout_of_grouped_intrinsics(mba, O, monkeypatch, solver):
    g = O.generate_groups(O.make_spec(num_cameras=24, num_points=1500, track_min=2, track_max=8, outlier_frac=0.05,
                                      seed=31), 3)
    const = np.zeros(24, np.uint8)
    const[2] = 1
    got = []
    for least in ("1", "1000000000"):
        print(f"layout: grouped solver {solver} least rows {least}", flush=True)
        monkeypatch.setenv("MBA_DEVICE_LAYOUT_MIN", least)
        p = mba.BAProblem(g["cam_init"].copy(), g["pt_init"].copy(), g["obs"], g["cam_idx"], g["pt_idx"], const,
                          intrinsics=g["intr_init"].copy(), intrinsic_index=g["intr_idx"],
                          intrinsic_constant=np.array([0, 1, 0], np.uint8),
                          intrinsic_subset=np.array([0x3E, 0, 0x38], np.uint8))
        s = mba.solve(p, mba.default_options(linear_solver=solver, huber_a=4.0, max_num_iterations=3))
        got.append([p.cameras, p.points, p.intrinsics, np.array(s.final_cost)])
    for x, y in zip(*got):
        np.testing.assert_array_equal(x, y)
