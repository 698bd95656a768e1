// Which logical block a workgroup takes.  constexpr functions, which hipcc
// compiles for both sides and a CPU test runs.
#pragma once

#include <cstdint>

namespace mfp {

// Workgroup ids are dispatched round-robin over the XCDs (each with its own
// L2).  Remap so that XCD k works on one contiguous range of logical blocks:
// neighbouring rows (and the x entries they share) stay in one L2.
constexpr uint32_t xcd_block(uint32_t b, uint32_t nb)
{
  constexpr uint32_t X = 8;
  if (nb < X * 4) return b;
  const uint32_t xcd = b % X, idx = b / X, q = nb / X, rem = nb % X;
  return xcd < rem ? xcd * (q + 1) + idx : rem * (q + 1) + (xcd - rem) * q + idx;
}

// The same in runs of 1 << run logical blocks: XCD k takes runs k, k + 8, ...
// Where the cost of a block differs along the range (a batch of matrices of
// several kinds), one contiguous range per XCD leaves the XCDs with the cheap
// ones idle at the end; a run still is long enough for its rows to share x.
constexpr uint32_t xcd_runs(uint32_t b, uint32_t nb, uint32_t run)
{
  const uint32_t w = 8u << run, at = b & ~(w - 1u);
  return at + xcd_block(b - at, (w < nb - at ? w : nb - at));
}

// xcd_runs, but each XCD begins with its runs an eighth of the grid after the
// one before and goes round: the XCDs are in different parts of the batch at a
// time, as with one range each, and still get an even share of every part.
constexpr uint32_t xcd_runs_turned(uint32_t b, uint32_t nb, uint32_t run)
{
  const uint32_t w = 8u << run, at = b & ~(w - 1u), m = nb >> (run + 3u); // m whole rounds of 8 runs
  uint32_t g = b >> (run + 3u);
  if (g >= m) return at + xcd_block(b - at, (w < nb - at ? w : nb - at));
  g += (b & 7u) * m / 8u; // below 2^29
  if (g >= m) g -= m;
  return (g << (run + 3u)) + xcd_block(b - at, w);
}

} // namespace mfp
