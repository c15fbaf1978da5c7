"""mba_evaluate_noalloc at the edges of its evaluation kernel: a wave's tile of
64 observations, a block's 256, remainders of both; 64 cameras (the table
formed by each block) and 65 (a launch of its own); outputs that are only
8-byte aligned.  Against the FP64 oracle.

Tolerances: FP64 values are sums of at most ~20 products of numbers of the
output's own size, each rounded once: 1e-12 of the array's largest entry
leaves a factor of ~200.  FP32 (mixed): the same count at 2^-24 relative to
the terms (the pixel scale, at most ~700, for residuals; the array's largest
entry for Jacobians): 2e-6.
"""
import numpy as np
import pytest

from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


def _scene(O, ncam, n):
    d = O.generate(O.make_spec(num_cameras=ncam, num_points=max(4, n // 2 + 2), track_min=2, track_max=4, seed=7 + n))
    cut = slice(0, n)
    return dict(d, obs=d["obs"][cut].copy(), cam_idx=d["cam_idx"][cut].copy(), pt_idx=d["pt_idx"][cut].copy())


@pytest.mark.parametrize("precision,tol", [(0, 1e-12), (1, 2e-6)])
@pytest.mark.parametrize("ncam,n,shift", [(64, 1, 0), (64, 63, 1), (65, 64, 1), (64, 65, 0), (65, 255, 0), (64, 257, 1),
                                          (65, 1029, 0)])
def test_evaluate_edges_match_oracle(mba, O, precision, tol, ncam, n, shift):
    d = _scene(O, ncam, n)
    npt = d["pt_init"].shape[0]
    h = _Hip(mba)
    st = h.stream()
    print(f"evaluate edges: {ncam} cameras {n} observations shift {shift} precision {precision}", flush=True)
    try:
        args = [h.put(d[k], t) for k, t in (("cam_init", np.float64), ("pt_init", np.float64), ("obs", np.float64),
                                            ("cam_idx", np.int32), ("pt_idx", np.int32))]
        # One value of padding before (shift) and after each output.
        out = {k: h.put(np.full(n * w + 2, -7.0), np.float64) for k, w in (("r", 2), ("jc", 18), ("jp", 6), ("c", 1))}
        off = 8 * shift
        mba.evaluate_noalloc(ncam, npt, n, *args, out["r"] + off, out["jc"] + off, out["jp"] + off, out["c"],
                             precision=precision, huber_a=4.0, stream=st)
        h.sync(st)
        got = {k: h.get(out[k], n * w + 2, np.float64) for k, w in (("r", 2), ("jc", 18), ("jp", 6), ("c", 1))}
    finally:
        h.close(st)
    ro, jco, jpo, _ = O.evaluate(O.Scene(d))
    for k, ref in (("r", ro), ("jc", jco), ("jp", jpo)):
        ref = np.asarray(ref).reshape(-1)
        scale = 700.0 if k == "r" else np.abs(ref).max()
        np.testing.assert_allclose(got[k][shift:shift + ref.size], ref, rtol=0, atol=tol * scale)
        assert (np.delete(got[k], np.arange(shift, shift + ref.size)) == -7.0).all(), k  # nothing written beside
    s = (ro.reshape(-1, 2) ** 2).sum(1)
    cost = np.where(s > 16.0, 4.0 * np.sqrt(s) - 8.0, 0.5 * s).sum()
    # d cost / d r <= 4 px per residual component at the Huber threshold.
    assert abs(got["c"][0] - cost) <= 1e-12 * cost + 8.0 * n * tol * 700.0
