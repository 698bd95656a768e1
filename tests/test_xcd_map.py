"""csrc/xcd_map.h on the CPU: every map of workgroups to logical blocks takes
each block once, and an XCD's blocks come in the runs that it promises."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "xcd_map.h"
#include <cstdio>
#include <cstdlib>
#include <vector>

using map_t = uint32_t (*)(uint32_t, uint32_t, uint32_t);

static void once(const char *name, map_t f, uint32_t nb, uint32_t run)
{
  std::vector<char> seen(nb, 0);
  for (uint32_t b = 0; b < nb; b++) {
    const uint32_t l = f(b, nb, run);
    if (l >= nb || seen[l]) {
      std::fprintf(stderr, "%s nb %u run %u: workgroup %u -> %u\n", name, nb, run, b, l);
      std::exit(1);
    }
    seen[l] = 1;
  }
}

int main()
{
  std::vector<uint32_t> sizes;
  for (uint32_t nb = 1; nb < 700; nb++) sizes.push_back(nb);
  for (uint32_t base : {1024u, 4096u, 8192u, 65536u, 100000u})
    for (int d = -9; d <= 9; d++) sizes.push_back(base + d);
  for (uint32_t nb : sizes)
    for (uint32_t run : {0u, 1u, 2u, 3u, 4u, 6u, 10u, 28u}) {
      once("runs", mfp::xcd_runs, nb, run);
      once("turned", mfp::xcd_runs_turned, nb, run);
    }
  // turned: an XCD's blocks of a whole round are 1 << run consecutive ones,
  // and it begins with the round that its eighth of the grid starts with
  const uint32_t nb = 40 * 128 + 5, run = 4, w = 128, m = 40;
  for (uint32_t x = 0; x < 8; x++)
    for (uint32_t g = 0; g < m; g++)
      for (uint32_t i = 0; i < 16; i++) {
        const uint32_t want = (g + x * m / 8) % m * w + x * 16 + i;
        if (mfp::xcd_runs_turned(g * w + i * 8 + x, nb, run) != want) return 1;
      }
  std::puts("ALL OK");
}
"""


def test_maps_take_every_block_once(tmp_path):
    src, exe = tmp_path / "check.cpp", str(tmp_path / "check")
    src.write_text(SOURCE)
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O2", "-Wall", "-Wextra",
                        "-I" + os.path.join(ROOT, "matrix_format_performance_amd", "csrc"), str(src), "-o", exe],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stderr[-2000:]
