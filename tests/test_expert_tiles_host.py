"""Which tiles the workgroups of the experts' large products take (csrc/expert_tiles.h), walked on the host as the kernel walks them: every tile of the
experts once or in both its halves, every tile with few rows and every tile of a shared expert once, and nothing else."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "minivllm_amd", "csrc")
PROGRAM = r"""
#include "expert_tiles.h"
#include <cstdio>
#include <random>
#include <vector>
using namespace mvllm;

int main() {
  std::mt19937 rng(7);
  auto below = [&](int n) { return (int)(rng() % (unsigned)n); };
  long halves = 0, several = 0, joined = 0;
  for (int turn = 0; turn < 30000; ++turn) {
    const int n_tiles = 1 + below(turn % 3 == 0 ? 40 : 9), whole = below(turn % 2 ? 130 : 20), rest = below(3) ? below(12) : 0;
    const int sh_rows = below(3) == 0 ? 0 : 1 + below(turn % 5 == 0 ? 40 : 6), sh_n = sh_rows ? 1 + below(turn % 7 == 0 ? 40 : 12) : 0;
    // workgroups per XCD as the host has them: the large form's, or one for every tile
    const int all = ((whole + rest + 1) * n_tiles + 7) / 8 + 1 + n_tiles + (sh_rows * sh_n + 7) / 8;
    const int groups = below(4) == 0 || all < kLargeGroups ? all : kLargeGroups;
    const int units = sh_rows && groups == kLargeGroups ? 1 + below(4) : 1;
    std::vector<int> taken((whole + rest) * n_tiles, 0), shared(sh_rows * sh_n, 0);         // a whole tile 3, its halves 1 and 2
    for (int xcd = 0; xcd < 8; ++xcd) {
      const LargeShare share(n_tiles, whole, rest, sh_rows, sh_n, units, xcd, groups);
      for (int group = 0; group < groups; ++group) {
        TilePlace t;
        int steps = 0;
        for (int j = group; share.find(j, t); j += groups * (t.shared ? units : 1)) {
          if (++steps > 100000) return printf("endless: turn %d\n", turn), 1;
          if (t.shared) {
            if (t.tile < 0 || t.tile >= sh_rows || t.n_tile < 0 || t.n_tile >= sh_n || t.half >= 0) return printf("shared place: turn %d\n", turn), 1;
            shared[t.tile * sh_n + t.n_tile] += 1;
            joined += units > 1;
            continue;
          }
          if (t.tile < 0 || t.tile >= whole + rest || t.n_tile < 0 || t.n_tile >= n_tiles || (t.half >= 0 && t.tile >= whole))
            return printf("place: turn %d\n", turn), 1;
          int& at = taken[t.tile * n_tiles + t.n_tile];
          const int part = t.half < 0 ? 3 : 1 << t.half;
          if (at & part) return printf("twice: turn %d\n", turn), 1;
          at |= part;
          halves += t.half >= 0;
        }
        several += steps > 1;
      }
    }
    for (int at : taken) if (at != 3) return printf("left out: turn %d\n", turn), 1;
    for (int at : shared) if (at != 1) return printf("shared %d times: turn %d\n", at, turn), 1;
  }
  if (halves < 10000 || several < 10000 || joined < 10000) return printf("cases: %ld %ld %ld\n", halves, several, joined), 1;
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not installed")
def test_every_tile_is_taken_once(tmp_path):
    source, program = tmp_path / "tiles.hip", tmp_path / "tiles"
    source.write_text(PROGRAM)
    subprocess.run(["hipcc", "--offload-host-only", "-O2", "-std=c++17", "-I" + CSRC, str(source), "-o", str(program)], check=True, capture_output=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout
