"""Memory kept between contexts: it goes back to the system on request, and what
a context finds in a used block (another size, layout or precision, a creation
that failed, another thread's problem) does not reach its results."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(O, ncam, npt, seed):
    d = O.generate(O.make_spec(num_cameras=ncam, num_points=npt, track_min=2, track_max=min(8, ncam), seed=seed))
    return {k: np.array(v) for k, v in d.items() if k in ("cam_init", "pt_init", "obs", "cam_idx", "pt_idx")}


def _solve(mba, d, **kw):
    p = mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), d["obs"], d["cam_idx"], d["pt_idx"])
    s = mba.solve(p, mba.default_options(max_num_iterations=3, **kw))
    return [p.cameras, p.points, np.array(s.final_cost)]


def _jobs(mba, O):
    """Solves of different sizes, solvers and precisions."""
    small, mid, large = _scene(O, 12, 300, 1), _scene(O, 40, 4000, 2), _scene(O, 120, 30000, 3)
    return [lambda: _solve(mba, large, linear_solver=mba.IMPLICIT_SCHUR_PCG, precision=mba.PRECISION_MIXED),
            lambda: _solve(mba, small),
            lambda: _solve(mba, mid, huber_a=4.0),
            lambda: _solve(mba, large),
            lambda: _solve(mba, small, linear_solver=mba.IMPLICIT_SCHUR_PCG),
            lambda: _solve(mba, mid, precision=mba.PRECISION_MIXED)]


def _failing(mba, O):
    """A context refused while it is built: SCHUR_JACOBI, a camera that sees a
    point twice (with the device layout, after its arrays are on the device)."""
    d = _scene(O, 30, 2000, 4)
    o = mba.default_options(linear_solver=mba.IMPLICIT_SCHUR_PCG, preconditioner=mba.PRECOND_SCHUR_JACOBI)
    twice = [np.concatenate([d[k], d[k][:1]]) for k in ("obs", "cam_idx", "pt_idx")]
    with pytest.raises(mba.MbaError):
        mba.Context(mba.BAProblem(d["cam_init"].copy(), d["pt_init"].copy(), *twice), o)


def test_cached_memory_goes_back_to_the_system(mba, O):
    import torch
    d = _scene(O, 200, 100000, 5)
    _solve(mba, d)
    before = torch.cuda.mem_get_info()[0]
    mba.release_cached_memory()
    # The observations alone (FP64, two orders) and S with its factor.
    least = 2 * 16 * len(d["obs"]) + 2 * 8 * (9 * 200) ** 2
    assert torch.cuda.mem_get_info()[0] - before > least
    mba.release_cached_memory()  # nothing left
    _solve(mba, d)


@pytest.mark.parametrize("least", ["1", "1000000000"])
def test_results_do_not_depend_on_what_a_block_held(mba, O, monkeypatch, least):
    monkeypatch.setenv("MBA_DEVICE_LAYOUT_MIN", least)
    jobs = _jobs(mba, O)
    fresh = []
    for job in jobs:
        mba.release_cached_memory()
        fresh.append(job())
    for order in ((0, 1, 2, 3, 4, 5), (5, 3, 1, 4, 0, 2), (2, 2, 0, 4, 3, 5)):
        for k in order:
            print(f"memory: layout {least} job {k}", flush=True)
            _failing(mba, O)
            for x, y in zip(jobs[k](), fresh[k]):
                np.testing.assert_array_equal(x, y)


def test_contexts_of_two_threads_share_the_memory(mba, O):
    jobs = _jobs(mba, O)
    want = [job() for job in jobs]
    got, errors = {}, []

    def work(first):
        try:
            for k in range(first, first + 2 * len(jobs)):
                got[first, k] = jobs[k % len(jobs)]()
                if k % 5 == 4:
                    mba.release_cached_memory()
        except Exception as e:  # reported by the test's thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(f,)) for f in (0, 3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for (_, k), out in got.items():
        for x, y in zip(out, want[k % len(jobs)]):
            np.testing.assert_array_equal(x, y)
