"""The rows of a ring that the prompt kernel of windowed attention reads: its own index functions, compiled for the host, over all places of a step in a ring."""
import os
import subprocess

from poptransformer_amd import build

PROGRAM = r"""
#include "ring.h"
#include <cstdio>
constexpr int KEYS = 64;

template <int DT>
static int check() {
  typedef KeyPairs<KEYS, DT * 4> Items;                        // a head of 32 * DT features in pieces of eight
  for (int idx = 0; idx < 256 * Items::PER_THREAD; ++idx) {
    const int pair = Items::pair(idx), piece = Items::piece(idx);
    if (idx < Items::ITEMS && pair * (DT * 4) + piece != idx) return printf("DT %d: item %d is pair %d, piece %d\n", DT, idx, pair, piece);
    for (int t = 0; t < 2; ++t) {
      const int k = pair * 2 + t;
      for (int len = 1; len <= 200; ++len)
        for (int first = 0; first < len; ++first)
          for (int ahead : {0, 1, 5, 62, 63, 64, 65, 127, 128, 500}) {       // the last position, behind the step's first
            const int jt = first + 3 * len, last = jt + ahead, row = ring_row<KEYS>(first, jt, k, last, len);
            const int want = (jt + k < last ? jt + k : last) % len;
            if (row < 0 || row >= len || row != want) return printf("DT %d: item %d, key %d of a step at %d of %d, last %d: row %d, not %d\n", DT, idx, k, first, len, last, row, want);
          }
    }
  }
  return 0;
}

int main() { return check<1>() || check<2>() || check<3>() || check<4>() || check<8>(); }
"""


def test_no_read_leaves_the_ring(tmp_path):
    source, program = tmp_path / "ring.hip", tmp_path / "ring"
    source.write_text(PROGRAM)
    subprocess.run([build._hipcc(), "--cuda-host-only", "-O2", "-std=c++17", "-I", os.path.join(build.CSRC, "hybrid"), str(source), "-o", str(program)], check=True, timeout=300)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout
