"""The frame window of the action branches' attention, checked on the CPU.

The kernels take it from ``csrc/hier_window.h``.  This test compiles that
header with g++ and UndefinedBehaviorSanitizer and compares it with the rule
it states (in 64 bits) over frames of every size: small ones on both sides of
0, the ends of an int, unbounded windows and windows of every length.
"""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "multics_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <vector>
#include "hier_window.h"
int main() {
  std::vector<int> frames;
  for (int f = -13; f <= 40; ++f) frames.push_back(f);
  for (int f : {100, 4095, 1 << 20, (1 << 30) + 7, INT_MAX - 40, INT_MAX - 1, -(1 << 20),
                INT_MIN + 40, INT_MIN + 1, INT_MIN}) frames.push_back(f);
  long seen = 0;
  for (int n_block : {1, 2, 3, 7, 1 << 20, INT_MAX})
    for (int w : {-1, 1, 2, 5, 21, 1 << 20, INT_MAX})
      for (int qf : frames) {
        hier::Window win;
        win.init(qf, n_block, w);
        if (win.sees(INT_MAX)) { printf("FAIL no key qf=%d n=%d w=%d\n", qf, n_block, w); return 1; }
        if (!win.sees(qf)) { printf("FAIL own qf=%d n=%d w=%d\n", qf, n_block, w); return 1; }
        for (int kf : frames) {
          const bool want = kf / n_block <= qf / n_block &&
                            (w < 0 || (int64_t)qf - kf < w);
          seen += want;
          if (win.sees(kf) != want) {
            printf("FAIL qf=%d kf=%d n=%d w=%d\n", qf, kf, n_block, w); return 1;
          }
        }
      }
  printf(seen > 1000 ? "OK\n" : "FAIL none\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_window_is_the_rule(tmp_path):
    src = tmp_path / "window.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "window"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined",
                    "-fno-sanitize-recover=undefined", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "OK", res.stdout + res.stderr
