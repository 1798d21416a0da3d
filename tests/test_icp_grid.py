"""Blocks of the tracking kernels by image size (openfusion_amd/csrc/kf_icp_grid.hpp), built
for the host: a step's slots cover the image; the single-launch form, whose blocks all have to
be on the chip at once, never takes more than one block per slot, nor, where two or more calls
fit 256 compute units that way, more than one per three pixels a thread of the finest level
and one pixel a thread of the others."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROG = r"""
#include <cstdio>
#include "kf_icp_grid.hpp"
int main() {
  for (int p = 256; p <= 8192 * 8192; p = p < 2000000 ? p + 61 : p + p / 7)
    for (int level = 0; level < 3; ++level)
      std::printf("%d %d %d %d %d\n", p, level, kf::kShapePixels[kf::step_shape(p)], kf::step_blocks(p, 1024),
                  kf::chain_blocks(p, level, 1024));
}
"""


def test_blocks_by_image_size():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        with open(src, "w") as f:
            f.write(PROG)
        subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{ROOT}/openfusion_amd/csrc", src, "-o", exe], check=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    for row in out.splitlines():
        pixels, level, shape, step, chain = map(int, row.split())
        assert step == min(-(-pixels // shape), 1024)
        few = -(-pixels // (512 * (3 if level == 0 else 1)))
        assert 1 <= chain <= step
        if few <= 128:
            assert chain <= few
