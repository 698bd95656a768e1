// Device helper shared by the converters and the selector's features.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfp {

// Rows of a tile of ROWS_TILE consecutive entries.  Given a row at or before
// the first entry's (one wave finds it with a 64-way search, one load per step
// where a binary search takes six, or it is the tile before's last row), each
// later row's number goes to its first entry in LDS, and a running maximum
// gives every entry its row.  A tile with far more rows than entries (long
// runs of empty rows) searches per entry instead.
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

// the same for a workgroup: its first wave searches, sh holds one word
__device__ __forceinline__ uint32_t block_row_of(const uint32_t *__restrict__ rp, uint32_t rows, uint32_t e,
                                                 uint32_t *sh)
{
  if (threadIdx.x < 64) {
    const uint32_t r = wave_row_of(rp, rows, e);
    if (threadIdx.x == 0) *sh = r;
  }
  __syncthreads();
  return *sh;
}

// row[k] = the row of entry t0 + ROWS_I threadIdx.x + k (entries at or past
// t1: of some entry of the tile).  t0 < t1 <= t0 + ROWS_TILE; rp[first] <= t0,
// and every row after first starts at t0 or later; sh_mark holds ROWS_TILE
// words and sh 4.
__device__ __forceinline__ void tile_rows(const uint32_t *__restrict__ rp, uint32_t rows, uint32_t first, uint32_t t0,
                                          uint64_t t1, uint32_t *sh_mark, uint32_t *sh, uint32_t (&row)[ROWS_I])
{
  constexpr uint32_t PER = 4; // rows per lane and step
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t m = (uint32_t)(t1 - t0);
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) sh_mark[k * ROWS_T + t] = 0;
  __syncthreads();
  // rows first + 1 .. that start inside the tile; of rows that start at the
  // same entry the last holds it
  for (uint64_t base = (uint64_t)first + 1;; base += ROWS_T * PER) {
    if (base - first > 16u * ROWS_TILE) {
      // the row of each entry by binary search from first on
#pragma unroll
      for (uint32_t k = 0; k < ROWS_I; k++) {
        const uint32_t e = t0 + min(t * ROWS_I + k, m - 1u);
        uint32_t lo = first, hi = rows;
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
    uint32_t p[PER];
#pragma unroll
    for (uint32_t q = 0; q < PER; q++) p[q] = rp[min(base + q * ROWS_T + t, (uint64_t)rows)];
    bool more = true;
#pragma unroll
    for (uint32_t q = 0; q < PER; q++) {
      const uint64_t r = base + q * ROWS_T + t;
      const bool in = r < rows && p[q] < t1;
      if (in) atomicMax(&sh_mark[p[q] - t0], (uint32_t)(r - first));
      more = more && in;
    }
    if (!__syncthreads_and(more)) break; // row starts only grow
  }
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
