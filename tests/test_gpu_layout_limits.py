"""The device-built layout against the host-built one where its rules change:
tracks at the longest one it takes and one beyond, more cameras than a
workgroup counts in LDS (one problem, grouped intrinsics, a batch whose
workgroups meet a short or a long range of cameras), camera-major rows split by
point ranges and the split given up when most rows belong to constant cameras,
and a camera with no more points than a point has cameras.  The values must be
the host layout's bit for bit; the preprocessing's trace tells which layout was
used."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("cam_init", "pt_init", "obs", "cam_idx", "pt_idx")


def _scene(O, ncam, npt, tmin, tmax, seed):
    d = O.generate(O.make_spec(num_cameras=ncam, num_points=npt, track_min=tmin, track_max=tmax, outlier_frac=0.05,
                               seed=seed))
    return {k: np.array(d[k]) for k in KEYS}


def _long_track(O, rows):
    """Point 0 seen by `rows` cameras (the rows added to it: at the image
    centre; the loss bounds them)."""
    d = _scene(O, 600, 100000, 4, 8, 3)
    have = d["cam_idx"][d["pt_idx"] == 0]
    add = np.setdiff1d(np.arange(600), have)[:rows - len(have)].astype(np.int32)
    return dict(d, obs=np.vstack([d["obs"], np.zeros((len(add), 2))]), cam_idx=np.concatenate([d["cam_idx"], add]),
                pt_idx=np.concatenate([d["pt_idx"], np.zeros(len(add), np.int32)]))


def _variant(O, name):
    """(scene, constant cameras, whether the device layout takes it)"""
    if name.startswith("track"):
        rows = int(name[5:])
        d = _long_track(O, rows)
        assert np.bincount(d["pt_idx"]).max() == rows and np.bincount(d["cam_idx"]).min() > 520
        return d, None, rows <= 512
    if name == "many_cameras":
        d = _scene(O, 4200, 40000, 3, 6, 4)
        assert np.bincount(d["cam_idx"], minlength=4200).min() > 6
        return d, None, True
    if name == "split":
        return _scene(O, 64, 80000, 3, 6, 5), None, True
    if name == "split_given_up":
        const = np.ones(64, np.uint8)
        const[[5, 20, 21, 60]] = 0
        d = _scene(O, 64, 80000, 3, 6, 5)
        assert len(d["obs"]) >= 2 ** 18 > np.isin(d["cam_idx"], np.flatnonzero(const == 0)).sum()
        return d, const, True
    # A camera whose points are as many as the longest track.
    d = _scene(O, 40, 3000, 3, 6, 6)
    keep = np.ones(len(d["obs"]), bool)
    keep[np.flatnonzero(d["cam_idx"] == 11)[6:]] = False
    return dict(d, **{k: d[k][keep] for k in ("obs", "cam_idx", "pt_idx")}), None, False


def _both(mba, monkeypatch, capfd, name, device, run):
    """run() with the device layout from 1 row on, and with the host layout."""
    monkeypatch.setenv("MBA_TRACE_PREP", "1")
    got = []
    for least in ("1", "1000000000"):
        print(f"layout limits: {name} least rows {least}", flush=True)
        monkeypatch.setenv("MBA_DEVICE_LAYOUT_MIN", least)
        capfd.readouterr()
        got.append(run())
        err = capfd.readouterr().err
        assert ("layout (device)" in err) == (device and least == "1")
        assert ("rows by point (device)" in err) == (least == "1")
    for x, y in zip(*got):
        assert np.all(np.isfinite(x))
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("name", ["track511", "track512", "track513", "many_cameras", "split", "split_given_up",
                                  "weak_camera"])
@pytest.mark.parametrize("precision", [0, 1])
def test_device_layout_at_its_limits(mba, O, monkeypatch, capfd, name, precision):
    d, const, device = _variant(O, name)

    def run():
        o = mba.default_options(precision=precision, linear_solver=mba.IMPLICIT_SCHUR_PCG, huber_a=4.0,
                                max_num_iterations=2)
        p = mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"], const)
        with mba.Context(p, o) as c:
            cost = c.lm_pass(1e4)
            b = c.read_schur()
            scale = c.read_scale()
        s = mba.solve(p, o)
        return [np.array(cost), *[b[k] for k in sorted(b)], *scale, p.cameras, p.points, np.array(s.final_cost)]

    _both(mba, monkeypatch, capfd, name, device, run)


def test_device_layout_of_many_grouped_cameras(mba, O, monkeypatch, capfd):
    g = O.generate_groups(O.make_spec(num_cameras=4200, num_points=40000, track_min=3, track_max=6,
                                      outlier_frac=0.05, seed=8), 5)
    # A point's degree counts its groups too: up to 6 cameras and 5 groups.
    assert np.bincount(g["cam_idx"], minlength=4200).min() >= 11

    def run():
        p = mba.BAProblem(g["cam_init"].copy(), g["pt_init"].copy(), g["obs"], g["cam_idx"], g["pt_idx"],
                          intrinsics=g["intr_init"].copy(), intrinsic_index=g["intr_idx"])
        s = mba.solve(p, mba.default_options(linear_solver=mba.IMPLICIT_SCHUR_PCG, huber_a=4.0, max_num_iterations=2))
        return [p.cameras, p.points, p.intrinsics, np.array(s.final_cost)]

    _both(mba, monkeypatch, capfd, "grouped", True, run)


@pytest.mark.parametrize("windows,cams,pts,unused", [(150, 30, 300, 0), (24, 5, 30, 600)])
def test_device_layout_of_a_batch_with_many_cameras(mba, O, monkeypatch, capfd, windows, cams, pts, unused):
    """More than 4,096 cameras in all: counted over the range of cameras that a
    workgroup's 256 points meet; with `unused` cameras without observations in
    front of each window's, that range is too long."""
    scenes = [_scene(O, cams, pts, 2, 3, 100 + k) for k in range(windows)]
    for d in scenes:
        assert np.bincount(d["cam_idx"], minlength=cams).min() > 3
        if unused:
            d["cam_init"] = np.vstack([np.repeat(d["cam_init"][:1], unused, 0), d["cam_init"]])
            d["cam_idx"] = (d["cam_idx"] + unused).astype(np.int32)
    assert sum(len(d["cam_init"]) for d in scenes) > 4096

    def run():
        probs = [mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"])
                 for d in scenes]
        # One iteration, and steps that no atomic sum reaches: one workgroup per
        # window for PCG (up to 64 cameras), the dense solver beyond.
        solver = mba.EXPLICIT_SCHUR if unused else mba.IMPLICIT_SCHUR_PCG
        sums = mba.solve_batched(probs, mba.default_options(linear_solver=solver, max_num_iterations=1, eta=1e-6))
        return [np.array([(s.num_e_blocks, s.num_f_blocks, s.termination_type) for s in sums]),
                np.concatenate([p.cameras for p in probs]), np.concatenate([p.points for p in probs])]

    _both(mba, monkeypatch, capfd, f"batch, {unused} unused", True, run)
