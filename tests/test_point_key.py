"""The device layout's point key: the widths of its fields, and that a problem
whose key does not fit 64 bits is left to the host's layout (the limit is asked
before anything is committed to the device's), not refused.  The engine's own
header, built for the host; such a problem itself (millions of windows) is
beyond a test."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(__file__), "..", "3dreconstruction_amd", "csrc")
MAIN = r"""
#include "mba_point_key.h"
#include <cstdio>
int main() {
  long long n;
  int W, deg, track;
  while (std::scanf("%lld %d %d %d", &n, &W, &deg, &track) == 4) {
    const mba::PointKey k(n, W, deg, track);
    std::printf("%d %d\n", k.bits(), (int)k.fits());
  }
}
"""


def test_point_key_widths_and_limit(tmp_path):
    (tmp_path / "main.cc").write_text(MAIN)
    exe = str(tmp_path / "a.out")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", exe, str(tmp_path / "main.cc")], check=True)
    calls = [(1, 1, 0, 1), (65536, 1, 6, 6), (4000000, 1, 50, 50), (6780000, 512, 40, 40),
             (2 ** 31 - 1, 1, 512, 512), (2 ** 31 - 1, 2 ** 13, 512, 512),  # 51, 64: the last that fits
             (2 ** 31 - 1, 2 ** 13 + 1, 512, 512), (2 ** 24, 2 ** 23, 512, 512)]
    out = subprocess.run([exe], input="\n".join("%d %d %d %d" % c for c in calls), capture_output=True, text=True,
                         check=True).stdout
    got = [tuple(int(x) for x in line.split()) for line in out.splitlines()]
    # Unobserved points need a length above the longest: all ones.
    want = [sum(v.bit_length() for v in (n, d, w - 1, t + 1)) for n, w, d, t in calls]
    assert got == [(b, int(b <= 64)) for b in want]
    assert [f for _, f in got] == [1, 1, 1, 1, 1, 1, 0, 0]


def test_the_limit_is_asked_before_the_device_layout_is_chosen():
    text = open(os.path.join(CSRC, "mba_engine.hip")).read()
    body = text[text.index("mba_status device_layout("):text.index("mba_status context_create(")]
    ask = re.search(r"if \(!PointKey\([^;]*\.fits\(\)\) return MBA_OK;", body)
    assert ask and body.index("lb.measure(") < ask.start() < body.index("c->grouped = grouped;")
