// Device helper shared by the converters and the selector's features.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfp {

// Rows of a tile of ROWS_TILE consecutive entries.  Two waves find the tile's
// first and last row with a 64-way search (one load per step where a binary
// search takes six), each row's number goes to its first entry in LDS, and a
// running maximum gives every entry its row.  A tile that spans far more rows
// than entries (long runs of empty rows) searches per entry instead.
constexpr uint32_t ROWS_T = 256, ROWS_I = 8, ROWS_TILE = ROWS_T * ROWS_I;

// largest r with rp[r] <= e, by one wave (every lane gets it); rp[0] <= e < rp[rows]
__device__ __forceinline__ uint32_t wave_row_of(const uint32_t *__restrict__ rp, uint32_t rows, uint32_t e)
{
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t lo = 0, hi = rows; // rp[lo] <= e < rp[hi]
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + 63u) / 64u; // >= 1
    const uint64_t at = (uint64_t)lo + (uint64_t)step * lane;
    const bool below = at < hi && rp[at] <= e; // lane 0: true
    const uint32_t k = (uint32_t)__popcll(__ballot(below)) - 1u; // a prefix of the lanes
    const uint32_t next = lo + step * k;
    hi = (uint32_t)min((uint64_t)hi, (uint64_t)next + step);
    lo = next;
  }
  return lo;
}

// row[k] = the row of entry t0 + ROWS_I threadIdx.x + k (entries at or past
// t1: the row of entry t1 - 1).  t0 < t1 <= t0 + ROWS_TILE; sh_mark holds
// ROWS_TILE words and sh 8.
__device__ __forceinline__ void tile_rows(const uint32_t *__restrict__ rp, uint32_t rows, uint32_t t0, uint64_t t1,
                                          uint32_t *sh_mark, uint32_t *sh, uint32_t (&row)[ROWS_I])
{
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t m = (uint32_t)(t1 - t0);
  if (wave < 2) {
    const uint32_t r = wave_row_of(rp, rows, wave ? t0 + (m - 1u) : t0);
    if (lane == 0) sh[4 + wave] = r;
  }
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) sh_mark[k * ROWS_T + t] = 0;
  __syncthreads();
  const uint32_t first = sh[4], last = sh[5];
  if (last - first > 16u * ROWS_TILE) {
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++) {
      const uint32_t e = t0 + min(t * ROWS_I + k, m - 1u);
      uint32_t lo = first, hi = last + 1;
      while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (rp[mid] <= e)
          lo = mid;
        else
          hi = mid;
      }
      row[k] = lo;
    }
    return;
  }
  // rows first + 1 .. last start inside the tile; of rows that start at the
  // same entry the last holds it
  for (uint32_t d = 1 + t; d <= last - first; d += ROWS_T) atomicMax(&sh_mark[rp[first + d] - t0], d);
  __syncthreads();
  uint32_t mx = 0;
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) {
    mx = max(mx, sh_mark[t * ROWS_I + k]);
    row[k] = mx;
  }
  uint32_t x = mx;
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x = max(x, y);
  }
  if (lane == 63) sh[wave] = x;
  uint32_t pre = __shfl_up(x, 1, 64);
  if (lane == 0) pre = 0;
  __syncthreads();
  for (uint32_t w = 0; w < wave; w++) pre = max(pre, sh[w]);
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) row[k] = first + max(pre, row[k]);
}

} // namespace mfp
