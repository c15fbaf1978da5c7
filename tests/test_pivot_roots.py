"""The FP64 pivots of the explicit Schur factors: the reciprocal square root from
the hardware's estimate (2^-24) is good to its last rounding (an IEEE square
root and division leave two).  The engine's own header, built for the host,
against 64-bit mantissas."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "3dreconstruction_amd", "csrc")
MAIN = r"""
#include "mba_rsqrt.h"
#include <cstdio>
int main() {
  double s, y;
  while (std::scanf("%lf %lf", &s, &y) == 2) {
    std::printf("%.17g\n", 2.0 * mba::refine_half_rsqrt(s, y));
  }
}
"""


@pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="needs an extended long double")
def test_pivot_root_is_good_to_rounding(tmp_path):
    (tmp_path / "main.cc").write_text(MAIN)
    exe = str(tmp_path / "a.out")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", CSRC, "-o", exe, str(tmp_path / "main.cc")],
                   check=True)
    rng = np.random.default_rng(5)
    # The scaled pivot is in [0.5, 2); ends and powers of two among the values.
    s = np.concatenate([rng.uniform(0.5, 2, 200000), [0.5, 1.0, np.nextafter(1, 0), np.nextafter(1, 2),
                                                      np.nextafter(2, 0)]])
    y = (1 + rng.uniform(-1, 1, len(s)) * 2.0 ** -24) / np.sqrt(s)
    text = "\n".join(f"{a:.17g} {b:.17g}" for a, b in zip(s, y))
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
    got = np.array([float(x) for x in out.split()])
    # Half a unit in the last place is at most 2^-53 of the value.
    rel = np.abs(got.astype(np.longdouble) * np.sqrt(s.astype(np.longdouble)) - 1)
    assert float(np.max(rel)) <= 1.001 * 2.0 ** -53
