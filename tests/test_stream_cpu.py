"""The batched kernel's place in its generator's stream (csrc/rng31.h) over more
moves than 32-bit positions hold: its ring entry, its refills and the
generator's front index stay those of 64-bit positions."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "mcgpu_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include "rng31.h"
using namespace mcgpu;

int main() {
  const int start = 17;
  StreamAt a;
  a.head = 31;
  long long pos = 0, head = 31;
  unsigned coin = 1;
  // 2^31 / 8 moves and then some
  for (long long move = 0; move < 275000000; move++) {
    if (stream_low(a) != (head < pos + 26) || (unsigned)a.pos % kRing != pos % kRing ||
        (unsigned)a.head % kRing != head % kRing || stream_front(a, start) != (start + pos) % 31 ||
        a.head - a.pos != head - pos) {
      std::printf("move %lld\n", move);
      return 1;
    }
    if (stream_low(a)) {
      a.head += 31;
      head += 31;
    }
    coin = coin * 1664525u + 1013904223u;
    const int draws = 8 + (int)(coin >> 31);
    stream_advance(a, draws);
    pos += draws;
  }
  return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a host compiler")
def test_positions_over_more_moves_than_32_bits_hold(tmp_path):
    src, exe = tmp_path / "stream.cpp", tmp_path / "stream"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
