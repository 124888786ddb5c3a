"""How a scan numbers its candidates over cells (csrc/scan_items.h): every
candidate in one place, a table that holds the pieces, and few free places
whatever the occupancies."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "mcgpu_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "scan_items.h"
using namespace mcgpu;

int main() {
  srand(5);
  for (int trial = 0; trial < 200000; trial++) {
    const int cells = 1 + rand() % 64, pass = 128 << rand() % 4;
    const int level = 1 + rand() % 40, fullest = 1 + rand() % (trial % 3 ? 3000 : 30);
    int n[64], largest = 0;
    long long sum = 0;
    for (int c = 0; c < cells; c++) {
      n[c] = rand() % 4 == 0 ? 0 : rand() % level;
      if (rand() % 12 == 0) n[c] = rand() % fullest;
      if (n[c] > largest) largest = n[c];
      sum += n[c];
    }
    const int w = scan_width(cells, largest, (int)sum, pass);
    long long entries = cells;
    if (w != largest) {
      entries = 0;
      for (int c = 0; c < cells; c++) entries += (n[c] + w - 1) / w;
    }
    const long long items = entries * w;
    bool ok = entries <= kScanEntries && items <= (long long)cells * largest && w <= largest;
    for (int c = 0; c < cells; c++) ok = ok && (w == largest ? n[c] <= w : w >= 1);
    // at most two items a candidate, beyond one pass, where the table has room
    if (cells <= 27) ok = ok && (items <= pass || items <= 2 * sum + cells);
    if (!ok) {
      std::printf("cells %d largest %d sum %lld pass %d width %d\n", cells, largest, sum, pass, w);
      return 1;
    }
  }
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a host compiler")
def test_items_follow_the_candidates(tmp_path):
    src, exe = tmp_path / "items.cpp", tmp_path / "items"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
