"""How the quantiser's workgroups are dealt out (csrc/mnb_quant_grid.h), compiled for the host.  No GPU needed."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "onnxruntime_amd" / "csrc"
PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "mnb_quant_grid.h"
int main() {
  // every tile once, whatever is left over among eight XCDs and in the last run
  for (int strips : {1, 2, 7, 8, 30, 129})
    for (int groups : {1, 2, 15, 16, 17, 31, 33, 100}) {
      const MnbQuantGrid g = mnb_quant_grid(strips, groups, 512, true);
      if (!g.ok || g.run != 16 || g.y != 1 || g.x != (unsigned)(strips * groups)) return 1;
      std::vector<int> seen(strips * groups);
      for (unsigned x = 0; x < g.x; ++x) {
        const MnbQuantTile t = mnb_quant_run_tile(x, g.x, strips, groups, g.run);
        if (t.strip < 0 || t.strip >= strips || t.group < 0 || t.group >= groups || seen[t.strip * groups + t.group]++) return 2;
      }
    }
  auto show = [](int64_t strips, int64_t groups, int threads, bool runs) {
    const MnbQuantGrid g = mnb_quant_grid(strips, groups, threads, runs);
    printf("%d %u %u %d\n", (int)g.ok, g.x, g.y, g.run);
  };
  show(1, 65536, 512, false);
  show(1, 65537, 512, false);
  show(64, 65536, 512, true);
  show(64, 65537, 512, true);
  show(128, 65535, 512, true);
  show(128, 65536, 512, true);
  show(512, 65535, 64, true);
}
"""


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    d = tmp_path_factory.mktemp("quant_grid")
    (d / "grid.cc").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", str(CSRC), "-o", str(d / "grid"), str(d / "grid.cc")],
                   check=True)
    return subprocess.run([str(d / "grid")], check=True, capture_output=True, text=True).stdout.split("\n")


def test_limits_of_a_launch(lines):
    """65536 groups along y are what the device takes; runs, all in x, stay below 2^32 threads or give way to the other order."""
    assert lines[:2] == ["1 1 65536 0", "0 1 65537 0"]
    assert lines[2:4] == [f"1 {64 * 65536} 1 16", f"0 {64 * 65537} 1 16"]
    assert lines[4:6] == [f"1 {128 * 65535} 1 16", "1 128 65536 0"]
    assert lines[6] == f"1 {512 * 65535} 1 16"
