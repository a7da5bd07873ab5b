"""CPU: the work split that a matvec launch is given (mfma_common.h).

The launch rules weigh a launch by the pairs (tile, stage) of its busiest
workgroup, so that count has to be what the kernels' schedule deals out: whole
tiles g, g + G, ..., then ranges of `width` leftover pairs.
"""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent
CSRC = REPO / "memory-aware-inference_amd" / "csrc"

PROGRAM = r"""
#include "mfma_common.h"
#include <cstdio>
using namespace sihip::mfma;
int main() {
  unsigned long checked = 0, split = 0;
  for (uint32_t cus : {255u, 256u})
    for (uint32_t waves : {4u, 8u, 12u})
      for (uint32_t tiles = 1; tiles < 2600; tiles += tiles % 256 < 8 ? 1 : 13)
        for (uint32_t parts = 1; parts <= 128; parts += parts < 24 ? 1 : 13) {
          const LaunchShape ls =
              launch_shape(tiles, parts, waves, sihip::kWorkspaceBytes, 1u, cus);
          const uint64_t G = ls.groups, X = ls.width, q = tiles / G;
          const uint64_t left = X ? (tiles - q * G) * parts : 0;
          uint64_t most = 0, touched = 0, dealt = 0;
          for (uint64_t g = 0; g < G; ++g) {
            const uint64_t a = std::min(g * X, left), b = std::min((g + 1) * X, left);
            const uint64_t whole = X ? q : g < tiles ? (tiles - 1 - g) / G + 1 : 0;
            const uint64_t own = whole + (b > a ? (b - 1) / parts - a / parts + 1 : 0);
            most = std::max(most, whole * parts + b - a);
            touched = std::max(touched, own);
            dealt += whole * parts + b - a;
          }
          ++checked;
          split += X != 0;
          if (most != ls.busiest || touched > ls.tiles_per_group || dealt != (uint64_t)tiles * parts) {
            std::printf("tiles %u parts %u waves %u cus %u: %lu pairs, said %lu\n", tiles, parts,
                        waves, cus, (unsigned long)most, (unsigned long)ls.busiest);
            return 1;
          }
        }
  std::printf("%lu %lu\n", checked, split);
  return 0;
}
"""


def test_busiest_workgroup(tmp_path):
    src, exe = tmp_path / "shape.hip", tmp_path / "shape"
    src.write_text(PROGRAM)
    subprocess.run(["/opt/rocm/bin/hipcc", "--cuda-host-only", "-std=c++17", "-O1",
                    "-Wno-unused-function", f"-I{REPO / 'include'}", f"-I{CSRC}", str(src), "-o",
                    str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
    checked, split = map(int, out.stdout.split())
    assert checked > 40000 and split > 4000
