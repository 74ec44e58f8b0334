"""Iterations and row offsets of the streaming sweeps (fall3d_amd/csrc/ads_rows.h,
plain C++), compiled for the host: every row that a line's iterations store
lies inside the line's array, up to the largest pitch that initialize accepts."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "ads_rows.h"
int main() {
  const int pf = 4, table_rows_before = 24;
  int lowest = 0;
  for (int half = 0; half < 2; ++half)
    for (int nst = 1; nst <= 4; nst += 3)
      for (int n = 2; n <= 1200; ++n) {
        // the largest pitch: whole 128-byte rows, n + 4 of them below 2^31 bytes
        const long long pitch = ((1ll << 31) - 1) / (n + 4) / 128 * 128;
        const f3d::StreamSpan s = f3d::stream_span(n, nst, pf, half != 0);
        if (s.last != n + 2 * nst + 1 || (s.last + 1 - s.first_block) % 16) return 1;
        if (s.first > 2 - pf || s.first <= -table_rows_before) return 2;
        if (s.first != s.first_block && (s.first != s.first_block + 8 || !half)) return 3;
        if (half && s.first + 8 <= 2 - pf && s.first == s.first_block) return 4;
        for (int t = s.first; t <= s.last; ++t) {
          const int row = t - 2 * nst;  // cell t - 2 nst - 1, row 0 is cell -1
          lowest = row < lowest ? row : lowest;
          const long long want = (row > 0 ? row : 0) * pitch;
          if ((long long)f3d::row_offset(row, (uint32_t)pitch) != want) return 5;
          if (want > (n + 1) * pitch) return 6;  // cell n is the last one stored
        }
        if (f3d::row_offset(s.last - 2 * nst, (uint32_t)pitch) != (uint32_t)((n + 1) * pitch)) return 7;
      }
  std::printf("%d\n", lowest);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_stored_rows_stay_inside_the_line(tmp_path):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-I", os.path.join(ROOT, "fall3d_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert int(r.stdout) < -16  # the span does reach far below the line
