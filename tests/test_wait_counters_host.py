"""The comparison of the waves' counters (nbg_types.h, as the kernels use it):
right across 2^31, where a signed comparison goes wrong, and across the wrap at
2^32, for every distance a ring allows.  Compiled for the host with the
optimisation that folds a signed `a - b < 0` into `a < b`."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nbodygradient.jl_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "nbg_types.h"
int main() {
  const uint32_t at[] = {0u, 1u, 100u, 0x7fffff00u, 0x7fffffffu, 0x80000000u, 0x80000010u, 0xffffff00u, 0xffffffffu};
  int bad = 0;
  for (uint32_t a : at)
    for (int d = -300; d <= 300; ++d)  // the counter is d ahead of the value waited for
      if (nbg::counter_reached(a + (uint32_t)d, a) != (d >= 0)) ++bad;
  // a wait's own course: the counter climbs to the value from a ring below
  for (uint32_t want = nbg::COUNTER_START; want != nbg::COUNTER_START + 1024u; ++want) {
    uint32_t have = want - 132u;
    int polls = 0;
    while (!nbg::counter_reached(have, want)) { ++have; ++polls; }
    if (polls != 132) ++bad;
  }
  std::printf("%d\n", bad);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_counters_across_their_wrap(tmp_path):
    src, exe = str(tmp_path / "c.cpp"), str(tmp_path / "c")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, src, "-o", exe], check=True)
    assert subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout.strip() == "0"
