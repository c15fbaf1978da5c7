"""A problem structure keeps the arrays it points at: another thread may give the
problem other arrays while a call runs on the structure (ctypes releases the
interpreter lock)."""
import gc
import weakref

import numpy as np

from conftest import ba_problem, grouped_problem

NAMES = ("cameras", "points", "observations", "camera_index", "point_index", "camera_constant", "intrinsics",
         "intrinsic_index", "intrinsic_constant", "intrinsic_subset")


def _refs(p):
    """Weak references to the problem's arrays, which the problem then loses."""
    refs = {n: weakref.ref(getattr(p, n)) for n in NAMES if getattr(p, n) is not None}
    for n in refs:
        a = getattr(p, n)
        setattr(p, n, np.array(a))
        del a
    gc.collect()
    return refs


def _own(p):
    for n in NAMES:
        if getattr(p, n) is not None:
            setattr(p, n, np.array(getattr(p, n)))
    return p


def test_a_structure_keeps_its_arrays(mba, O, tiny_scene):
    g = O.generate_groups(O.make_spec(num_cameras=6, num_points=40, track_min=2, track_max=4, seed=3), 2)
    for p in (_own(ba_problem(mba, tiny_scene, np.zeros(len(tiny_scene["cam_init"]), np.uint8))),
              _own(grouped_problem(mba, g, intr_const=np.zeros(2, np.uint8), subset=np.zeros(2, np.uint8)))):
        s = p._struct()
        refs = _refs(p)
        assert len(refs) >= 6 and all(r() is not None for r in refs.values())
        assert s.cameras == refs["cameras"]().ctypes.data
        del s
        gc.collect()
        assert all(r() is None for r in refs.values())


def test_a_batch_keeps_its_arrays_during_the_call(mba, tiny_scene, monkeypatch):
    problems = [_own(ba_problem(mba, tiny_scene)) for _ in range(3)]
    seen = []

    class Library:
        def mba_solve_batched(self, *a):
            refs = [r for p in problems for r in _refs(p).values()]
            seen.extend(r() is not None for r in refs)
            return 0

    monkeypatch.setattr(mba, "load_library", lambda: Library())
    o = mba.Options()
    mba.solve_batched(problems, o)
    assert len(seen) == 15 and all(seen)
