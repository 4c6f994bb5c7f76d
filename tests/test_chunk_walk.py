"""The keys that a workgroup of the chunk attention reads of gathered latent rows (csrc/mixers/chunk_walk.h, the arithmetic of
the kernel itself, built for the host) stay inside its sequence's rows, and are all that its queries see."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "chunk_walk.h"
using namespace mxs;
int main() {
  const int lengths[] = {1, 5, 16, 17, 40, 129}, kt = 32;
  long read = 0;
  for (int past = 0; past < 200; ++past)
    for (int window = 0; window < 100; ++window)
      for (int n : lengths)
        for (int per = 40; per <= 128; per += 88) {  // queries of a workgroup
          const int low = first_gathered(past, window), rows = past + n - low;
          for (int q0 = 0; q0 < n; q0 += per) {
            const int first = past + q0, last = past + (q0 + per < n ? q0 + per : n) - 1;
            const ChunkWalk w = chunk_walk(first, last, window, 0, kt);
            std::vector<char> seen(past + n + 1, 0);
            for (int it = 0; it < w.ntile; ++it)
              for (int page = 0; page < kt / kWalkPage; ++page) {
                const int key0 = w.start(it) + kWalkPage * page, left = gathered_left(key0, low, last);
                for (int r = 0; r < kWalkPage && r <= left; ++r) {
                  const int row = key0 + r - low;  // of this sequence's gathered rows
                  if (row < 0 || row >= rows) { printf("past %d window %d n %d: row %d of %d\n", past, window, n, row, rows); return 1; }
                  ++seen[key0 + r];
                  ++read;
                }
              }
            const int oldest = window > 0 && first - window + 1 > 0 ? first - window + 1 : 0;
            for (int j = oldest; j <= last; ++j)
              if (seen[j] != 1) { printf("past %d window %d n %d: key %d read %d times\n", past, window, n, j, seen[j]); return 1; }
          }
        }
  printf("OK %ld\n", read);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_reads_stay_inside_the_gathered_rows(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "csrc", "mixers"), str(src), "-o", str(exe)], check=True,
                   capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("OK"), r.stdout
