"""Index arithmetic of csrc/row_chunks.h near 2^32 entries (CPU only; the
library takes up to 2^32 - 1 entries, a size that no GPU test allocates)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "row_chunks.h"
#include <cstdio>
#include <cstdlib>

int main()
{
  const uint64_t ends[] = {0, 1, 959, 960, 961, 1984, 4000, 70000, (1ull << 32) - 1985, (1ull << 32) - 1984,
                           (1ull << 32) - 961, (1ull << 32) - 960, (1ull << 32) - 2, (1ull << 32) - 1};
  const uint64_t lengths[] = {0, 1, 2, 959, 960, 961, 1920, 1983, 1984, 1985, 3968, 3969, 50000, 1000003};
  const uint32_t chunks[] = {960, 1984};
  for (uint64_t e : ends)
    for (uint64_t len : lengths)
      for (uint32_t chunk : chunks) {
        if (len > e) continue;
        uint64_t at = e - len, calls = 0; // the next element to be covered
        mfp::for_row_chunks((uint32_t)at, (uint32_t)e, chunk, [&](uint32_t start, uint32_t n) {
          const bool last = at + n == e;
          if (start != at || n == 0 || n > chunk || (!last && n != chunk) || ++calls > len) {
            std::fprintf(stderr, "end %llu length %llu chunk %u: start %u n %u, expected start %llu\n",
                         (unsigned long long)e, (unsigned long long)len, chunk, start, n, (unsigned long long)at);
            std::exit(1);
          }
          at += n;
        });
        if (at != e) return 1;
      }
  std::puts("ALL OK");
}
"""


def test_row_chunks_up_to_the_last_entry(tmp_path):
    src, exe = tmp_path / "check.cpp", str(tmp_path / "check")
    src.write_text(SOURCE)
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Wextra",
                        "-I" + os.path.join(ROOT, "matrix_format_performance_amd", "csrc"), str(src), "-o", exe],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stderr[-2000:]
