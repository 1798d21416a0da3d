"""The parts of a one-thread-per-item launch (openfusion_amd/csrc/kf_launch.hpp), built for
the host: at every volume size that kf_volume_create takes, both voxel formats, the launches
that fill it cover its 16-byte vectors once, in order, each with fewer than 2^32 threads
(the limit of a HIP grid)."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROG = r"""
#include <cstdio>
#include "kf_launch.hpp"
int main() {
  for (size_t n = 8; n <= 2048; n += 8)
    for (size_t bytes = 4; bytes <= 8; bytes += 4) {
      const size_t items = n * n * n * bytes / 16;
      size_t next = 0, parts = 0;
      int bad = 0;
      kf::launch_items(items, [&](size_t first, size_t count, unsigned blocks) {
        const size_t threads = (size_t)blocks * kf::kItemThreads;
        bad |= first != next || count == 0 || threads < count || threads >= count + kf::kItemThreads || threads >> 32;
        next = first + count;
        ++parts;
        return 0;
      });
      std::printf("%zu %zu %d %zu\n", n, bytes, bad || next != items, parts);
    }
  // a launch that fails ends the sequence
  size_t calls = 0;
  const int st = kf::launch_items(3 * kf::kMaxLaunchItems, [&](size_t, size_t, unsigned) { return ++calls == 2 ? 7 : 0; });
  std::printf("fail %d %zu\n", st, calls);
}
"""


def test_volume_fill_launches():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        with open(src, "w") as f:
            f.write(PROG)
        subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{ROOT}/openfusion_amd/csrc", src, "-o", exe], check=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split("\n")
    rows = [tuple(map(int, r.split())) for r in out if r and not r.startswith("fail")]
    assert len(rows) == 2 * 256
    assert all(bad == 0 for _, _, bad, _ in rows)
    assert {(n, b): p for n, b, _, p in rows}[2048, 8] == 2  # 2^32 vectors
    assert "fail 7 2" in out
