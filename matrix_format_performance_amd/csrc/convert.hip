// Device-side matrix converters.
//
// The reference builds every layout on the host (common/matrix_converter.cpp,
// common/scoo_matrix_class.cpp, gpu/csr_adaptive_spmv.cu:180-240).  Here each
// layout is built by HIP kernels in HBM; the results are bit-identical to the
// reference's host algorithms (ties in triplets->CSR keep input order).
#include "entry_rows.h"
#include "mfp_internal.h"
#include "wave64.h"

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

namespace mfp {

// Device allocations freed on every return path unless released.
struct device_temps {
  std::vector<void *> held;
  bool idle = false; // their one stream was waited for
  int alloc(void **p, size_t bytes)
  {
    const int st = dmalloc(p, bytes);
    idle = false; // work on it follows
    if (st == MFP_OK) held.push_back(*p);
    return st;
  }
  void release(void *p)
  {
    for (void *&q : held)
      if (q == p) q = nullptr;
  }
  // waits for the stream that alone uses them
  int settle(hipStream_t s)
  {
    MFP_HIP(hipStreamSynchronize(s));
    idle = true;
    return MFP_OK;
  }
  ~device_temps()
  {
    const free_scope scope(idle);
    for (void *q : held) dfree(q);
  }
};

// ---------------------------------------------------------------------------
// Exclusive scan of u32: tile sums, one workgroup scans those, then every
// tile scans itself from its offset (8 bytes read and 4 written per element,
// three launches; one for a single tile).
// ---------------------------------------------------------------------------
constexpr uint32_t SCAN_T = 256, SCAN_I = 16, SCAN_TILE = SCAN_T * SCAN_I;

// Exclusive prefix of v over a workgroup of T lanes; *total (may be null)
// gets the sum.  sh holds T / 64 words.
template <uint32_t T>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *sh, uint32_t *total)
{
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint32_t pre = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < T / 64; w++) {
    const uint32_t s = sh[w];
    if (w < wave) pre += s;
    all += s;
  }
  if (total) *total = all;
  __syncthreads(); // sh may be written again
  return pre + x - v;
}

__global__ __launch_bounds__(SCAN_T) void k_scan_sums(const uint32_t *__restrict__ in, uint64_t n,
                                                      uint32_t *__restrict__ sums)
{
  __shared__ uint32_t sh[SCAN_T / 64];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
  uint32_t acc = 0;
#pragma unroll
  for (uint32_t k = 0; k < SCAN_I; k++) {
    const uint64_t i = base + k * SCAN_T + threadIdx.x;
    acc += i < n ? in[i] : 0u;
  }
  uint32_t total;
  (void)block_exclusive_scan<SCAN_T>(acc, sh, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// sums[0 .. m) to their exclusive scan, the total to sums[m]; one workgroup
__global__ __launch_bounds__(1024) void k_scan_offsets(uint32_t *__restrict__ sums, uint64_t m)
{
  __shared__ uint32_t sh[16];
  uint32_t carry = 0;
  for (uint64_t b = 0; b < m; b += 1024) {
    const uint64_t i = b + threadIdx.x;
    const uint32_t v = i < m ? sums[i] : 0u;
    uint32_t total;
    const uint32_t pre = block_exclusive_scan<1024>(v, sh, &total);
    if (i < m) sums[i] = carry + pre;
    carry += total;
  }
  if (threadIdx.x == 0) sums[m] = carry;
}

// offs: k_scan_offsets' result, or null for a single tile (whose total then
// goes to *total)
__global__ __launch_bounds__(SCAN_T) void k_scan_tiles(const uint32_t *in, uint32_t *out, uint64_t n,
                                                       const uint32_t *__restrict__ offs,
                                                       uint32_t *__restrict__ total)
{
  __shared__ uint32_t tile[SCAN_TILE + SCAN_TILE / 32]; // one word of padding per 32: lanes read SCAN_I apart
  __shared__ uint32_t sh[SCAN_T / 64];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
  const uint32_t t = threadIdx.x;
#pragma unroll
  for (uint32_t k = 0; k < SCAN_I; k++) {
    const uint32_t l = k * SCAN_T + t;
    tile[l + l / 32] = base + l < n ? in[base + l] : 0u;
  }
  __syncthreads();
  uint32_t loc[SCAN_I], acc = 0;
#pragma unroll
  for (uint32_t k = 0; k < SCAN_I; k++) {
    const uint32_t l = t * SCAN_I + k;
    loc[k] = acc;
    acc += tile[l + l / 32];
  }
  uint32_t all;
  const uint32_t pre = block_exclusive_scan<SCAN_T>(acc, sh, &all) + (offs ? offs[blockIdx.x] : 0u);
#pragma unroll
  for (uint32_t k = 0; k < SCAN_I; k++) {
    const uint32_t l = t * SCAN_I + k;
    tile[l + l / 32] = loc[k] + pre;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < SCAN_I; k++) {
    const uint32_t l = k * SCAN_T + t;
    if (base + l < n) out[base + l] = tile[l + l / 32];
  }
  if (!offs && t == 0) *total = all;
}

// In-place (in == out) is allowed.  total_out (host, may be null) gets in[0..n)
// summed.  Waits for the stream.
int exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint64_t n, hipStream_t s,
                       uint32_t *total_out)
{
  if (total_out) *total_out = 0;
  if (n == 0) return MFP_OK;
  const uint64_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
  device_temps tmp;
  uint32_t *sums = nullptr;
  MFP_CHECK(tmp.alloc((void **)&sums, (tiles + 1) * 4));
  if (tiles > 1) {
    k_scan_sums<<<(uint32_t)tiles, SCAN_T, 0, s>>>(in, n, sums);
    k_scan_offsets<<<1, 1024, 0, s>>>(sums, tiles);
    k_scan_tiles<<<(uint32_t)tiles, SCAN_T, 0, s>>>(in, out, n, sums, nullptr);
  } else {
    k_scan_tiles<<<1, SCAN_T, 0, s>>>(in, out, n, nullptr, sums + tiles);
  }
  MFP_HIP(hipGetLastError());
  if (total_out) MFP_HIP(hipMemcpyAsync(total_out, sums + tiles, 4, hipMemcpyDeviceToHost, s));
  MFP_CHECK(tmp.settle(s)); // sums is freed here
  return MFP_OK;
}

// ---------------------------------------------------------------------------
// Stable radix sort of (row, column, value) entries by (row, column), least
// significant digit first.  The values travel with the keys, so nothing is
// gathered at the end, and as every pass keeps the order of equal digits no
// input index is carried.  row may be any u32 whose bits above row_shift
// count (the column-sorted layout sorts by slice).
//   k_sort_count    digit counts of each tile (SORT_T ITEMS entries)
//   k_sort_offsets  one workgroup per digit: exclusive scan over the tiles
//   k_sort_scatter  ranks a tile's entries by digit (ballots inside a wave,
//                   LDS counts across waves), reorders them in LDS and
//                   writes each digit's run to its place
// Bound by the writes: 4096 entries make runs of 16 on average, so most lines
// are written by two tiles or more.  Tiles side by side are on one XCD (runs of
// 32 tiles) and so complete each other's lines in its L2, which is what lets a
// tile be this small, with three workgroups per CU to overlap the loads, the
// ranking and the stores.  11.7M FP32 entries, a pass of 281 MB: tiles dealt
// round robin 82 us (8192 entries) and 85 (4096), on one XCD 76 and 67; 3072
// entries 70, 2048 79; the first pass, which reads doubles, 115 -> 78; with
// runs of 64 tiles the same, of 16 or 256 and one range per XCD 2% slower.
// ---------------------------------------------------------------------------
constexpr uint32_t SORT_T = 512, SORT_W = SORT_T / 64, SORT_BINS = 256;
constexpr uint32_t SORT_RUN = 5; // log2 of the tiles an XCD takes in a row

struct sort_digit {
  uint32_t row_shift; // row bits below this do not take part
  uint32_t col_bits;  // columns are below 2^col_bits
  uint32_t shift, width; // the digit's place in (row >> row_shift) 2^col_bits + column
};

__device__ __forceinline__ uint32_t digit_of(const sort_digit &d, uint32_t row, uint32_t col)
{
  const uint64_t key = ((uint64_t)(row >> d.row_shift) << d.col_bits) | col;
  return (uint32_t)(key >> d.shift) & ((1u << d.width) - 1u);
}

// CHECK: also sets *bad when a row is not below rows or a column not below cols
template <uint32_t ITEMS, bool CHECK>
__global__ __launch_bounds__(SORT_T) void k_sort_count(const uint32_t *__restrict__ row,
                                                       const uint32_t *__restrict__ col, uint64_t n, sort_digit dg,
                                                       uint32_t rows, uint32_t cols, uint32_t ntiles,
                                                       uint32_t *__restrict__ hist, uint32_t *__restrict__ bad)
{
  __shared__ uint32_t cnt[SORT_BINS];
  const uint32_t t = threadIdx.x;
  if (t < SORT_BINS) cnt[t] = 0;
  __syncthreads();
  const uint32_t tile = xcd_runs(blockIdx.x, gridDim.x, SORT_RUN);
  const uint64_t base = (uint64_t)tile * (SORT_T * ITEMS);
  const bool need_row = CHECK || dg.shift + dg.width > dg.col_bits, need_col = CHECK || dg.shift < dg.col_bits;
  uint32_t r[ITEMS], c[ITEMS];
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const uint64_t i = min(base + k * SORT_T + t, n - 1);
    r[k] = need_row ? row[i] : 0u;
    c[k] = need_col ? col[i] : 0u;
  }
  bool out = false;
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++)
    if (base + k * SORT_T + t < n) {
      atomicAdd(&cnt[digit_of(dg, r[k], c[k])], 1u);
      if (CHECK) out = out || r[k] >= rows || c[k] >= cols;
    }
  if (CHECK && out) atomicOr(bad, 1u);
  __syncthreads();
  if (t < (1u << dg.width)) hist[(uint64_t)t * ntiles + tile] = cnt[t];
}

// row d of hist to its exclusive scan, its total to totals[d]
__global__ __launch_bounds__(1024) void k_sort_offsets(uint32_t ntiles, uint32_t *__restrict__ hist,
                                                       uint32_t *__restrict__ totals)
{
  __shared__ uint32_t sh[16];
  uint32_t *h = hist + (uint64_t)blockIdx.x * ntiles;
  uint32_t carry = 0;
  for (uint32_t b = 0; b < ntiles; b += 1024) {
    const uint32_t i = b + threadIdx.x;
    const uint32_t v = i < ntiles ? h[i] : 0u;
    uint32_t total;
    const uint32_t pre = block_exclusive_scan<1024>(v, sh, &total);
    if (i < ntiles) h[i] = carry + pre;
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// VI: the values' type as read (the first pass of a triplet sort rounds
// double values to the matrix's type), V: as moved and written
template <typename VI, typename V, uint32_t ITEMS>
__global__ __launch_bounds__(SORT_T, 6) void k_sort_scatter(const uint32_t *__restrict__ row,
                                                         const uint32_t *__restrict__ col,
                                                         const VI *__restrict__ val, uint64_t n, sort_digit dg,
                                                         uint32_t ntiles, const uint32_t *__restrict__ hist,
                                                         const uint32_t *__restrict__ totals,
                                                         uint32_t *__restrict__ orow, uint32_t *__restrict__ ocol,
                                                         V *__restrict__ oval)
{
  constexpr uint32_t TILE = SORT_T * ITEMS;
  __shared__ __align__(16) unsigned char buf_raw[TILE * (sizeof(V) > 4 ? sizeof(V) : 4)];
  __shared__ uint32_t cnt[SORT_W][SORT_BINS]; // entries of each digit in the waves before
  __shared__ uint32_t start[SORT_BINS];       // first slot of a digit's run in the tile
  __shared__ uint32_t glob[SORT_BINS];        // output position of the run, less start
  __shared__ uint32_t sh[SORT_W];
  uint32_t *buf = reinterpret_cast<uint32_t *>(buf_raw);
  V *vbuf = reinterpret_cast<V *>(buf_raw);
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t tile = xcd_runs(blockIdx.x, gridDim.x, SORT_RUN);
  const uint64_t base = (uint64_t)tile * TILE;
  const uint32_t m = (uint32_t)min((uint64_t)TILE, n - base); // entries of this tile
  // wave w holds entries w 64 ITEMS .. of the tile, 64 consecutive per item
  const uint32_t l0 = wave * 64u * ITEMS + lane;
  uint32_t r[ITEMS], c[ITEMS], pos[ITEMS];
  V v[ITEMS];
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const uint64_t i = base + min(l0 + k * 64u, m - 1u);
    r[k] = row[i];
    c[k] = col[i];
    v[k] = (V)val[i];
  }
#pragma unroll
  for (uint32_t b = 0; b < SORT_BINS / 64; b++) cnt[wave][b * 64u + lane] = 0;
  // only this wave touches its row of cnt until the barrier below
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const uint64_t below = lane ? ~0ull >> (64u - lane) : 0ull;
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const bool valid = l0 + k * 64u < m;
    const uint32_t d = digit_of(dg, r[k], c[k]);
    uint64_t peers = __ballot(valid);
    for (uint32_t b = 0; b < dg.width; b++) {
      const bool one = (d >> b) & 1u;
      const uint64_t ones = __ballot(one);
      peers &= one ? ones : ~ones;
    }
    const uint32_t before = cnt[wave][d];
    pos[k] = before + (uint32_t)__popcll(peers & below);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (valid && (peers & below) == 0) cnt[wave][d] = before + (uint32_t)__popcll(peers);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  __syncthreads();
  uint32_t mine = 0, tot = 0;
  if (t < SORT_BINS) {
#pragma unroll
    for (uint32_t w = 0; w < SORT_W; w++) {
      const uint32_t x = cnt[w][t];
      cnt[w][t] = mine;
      mine += x;
    }
    tot = t < (1u << dg.width) ? totals[t] : 0u;
  }
  const uint32_t st = block_exclusive_scan<SORT_T>(mine, sh, nullptr);
  const uint32_t gt = block_exclusive_scan<SORT_T>(tot, sh, nullptr);
  if (t < SORT_BINS) {
    start[t] = st;
    glob[t] = t < (1u << dg.width) ? gt + hist[(uint64_t)t * ntiles + tile] - st : 0u;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const uint32_t d = digit_of(dg, r[k], c[k]);
    pos[k] += start[d] + cnt[wave][d];
  }
  // slot order: rows, columns, then values through the same LDS
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++)
    if (l0 + k * 64u < m) buf[pos[k]] = r[k];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) r[k] = buf[min(k * SORT_T + t, m - 1u)];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++)
    if (l0 + k * 64u < m) buf[pos[k]] = c[k];
  __syncthreads();
  uint32_t to[ITEMS];
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const uint32_t j = k * SORT_T + t;
    c[k] = buf[min(j, m - 1u)];
    to[k] = glob[digit_of(dg, r[k], c[k])] + j;
    if (j < m) {
      orow[to[k]] = r[k];
      ocol[to[k]] = c[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++)
    if (l0 + k * 64u < m) vbuf[pos[k]] = v[k];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ITEMS; k++) {
    const uint32_t j = k * SORT_T + t;
    if (j < m) oval[to[k]] = vbuf[j];
  }
}

static uint32_t bit_length(uint32_t v)
{
  uint32_t b = 0;
  while (v) {
    b++;
    v >>= 1;
  }
  return b;
}

static uint32_t grid_for(uint64_t n, uint32_t bs = 256)
{
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + bs - 1) / bs, 1u << 16));
}

// The arrays of one side of the sort's ping-pong.
template <typename V>
struct sort_arrays {
  uint32_t *row = nullptr, *col = nullptr;
  V *val = nullptr;
};

// Sorts n >= 1 entries into `to`, using `via` between passes; the input is
// not written.  key_rows / cols bound (row >> row_shift) and the columns.
// bad (may be null): set when a row is not below rows or a column not below
// cols; the sort stays in bounds either way.
template <typename VI, typename V, uint32_t ITEMS>
static int sort_entries_t(const uint32_t *row, const uint32_t *col, const VI *val, uint64_t n, uint32_t row_shift,
                          uint64_t key_rows, uint32_t rows, uint32_t cols, const sort_arrays<V> &to,
                          const sort_arrays<V> &via, uint32_t *bad, hipStream_t s)
{
  const uint32_t col_bits = bit_length(cols ? cols - 1 : 0);
  const uint32_t bits = col_bits + bit_length(key_rows ? (uint32_t)(key_rows - 1) : 0);
  const uint32_t passes = std::max(1u, (bits + 7) / 8);
  const uint32_t width = std::max(1u, (bits + passes - 1) / passes); // as even as they come, at most 8
  const uint32_t ntiles = (uint32_t)((n + SORT_T * ITEMS - 1) / (SORT_T * ITEMS));
  device_temps tmp;
  uint32_t *hist = nullptr;
  MFP_CHECK(tmp.alloc((void **)&hist, ((uint64_t)ntiles + 1) * SORT_BINS * 4));
  uint32_t *totals = hist + (uint64_t)ntiles * SORT_BINS;
  for (uint32_t p = 0; p < passes; p++) {
    const sort_digit dg{row_shift, col_bits, p * width, width};
    const sort_arrays<V> &o = (passes - 1 - p) % 2 ? via : to; // the last pass lands in `to`
    const sort_arrays<V> &f = (passes - 1 - p) % 2 ? to : via;
    const uint32_t *fr = p ? f.row : row, *fc = p ? f.col : col;
    if (p == 0 && bad)
      k_sort_count<ITEMS, true><<<ntiles, SORT_T, 0, s>>>(fr, fc, n, dg, rows, cols, ntiles, hist, bad);
    else
      k_sort_count<ITEMS, false><<<ntiles, SORT_T, 0, s>>>(fr, fc, n, dg, rows, cols, ntiles, hist, nullptr);
    k_sort_offsets<<<1u << width, 1024, 0, s>>>(ntiles, hist, totals);
    if (p)
      k_sort_scatter<V, V, ITEMS><<<ntiles, SORT_T, 0, s>>>(fr, fc, f.val, n, dg, ntiles, hist, totals, o.row, o.col,
                                                            o.val);
    else
      k_sort_scatter<VI, V, ITEMS><<<ntiles, SORT_T, 0, s>>>(fr, fc, val, n, dg, ntiles, hist, totals, o.row, o.col,
                                                             o.val);
    MFP_HIP(hipGetLastError());
  }
  MFP_CHECK(tmp.settle(s)); // hist is freed here
  return MFP_OK;
}

template <typename VI, typename V>
static int sort_entries(const uint32_t *row, const uint32_t *col, const VI *val, uint64_t n, uint32_t row_shift,
                        uint64_t key_rows, uint32_t rows, uint32_t cols, const sort_arrays<V> &to,
                        const sort_arrays<V> &via, uint32_t *bad, hipStream_t s)
{
  // 4096 entries per tile, 2048 where those would be fewer than two per CU
  // (1.2M entries: 147 us against 157; 2M: 155 each)
  if (n >= (1u << 21))
    return sort_entries_t<VI, V, 8>(row, col, val, n, row_shift, key_rows, rows, cols, to, via, bad, s);
  return sort_entries_t<VI, V, 4>(row, col, val, n, row_shift, key_rows, rows, cols, to, via, bad, s);
}

// row_ptr[r] = entries in rows below r, from the entries' sorted rows
__global__ void k_row_starts(uint32_t rows, uint64_t n, const uint32_t *__restrict__ row, uint32_t *__restrict__ rp)
{
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r > rows) return;
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) / 2;
    if (row[mid] < r)
      lo = mid + 1;
    else
      hi = mid;
  }
  rp[r] = (uint32_t)lo;
}

template <typename V>
static int csr_from_triplets_t(uint32_t rows, uint32_t cols, uint64_t nnz, const uint32_t *tr_rows,
                               const uint32_t *tr_cols, const double *tr_vals, uint32_t *row_ptr, uint32_t *columns,
                               V *values, hipStream_t s)
{
  device_temps tmp;
  uint32_t *bad = nullptr;
  sort_arrays<V> to, via;
  to.col = columns;
  to.val = values;
  MFP_CHECK(tmp.alloc((void **)&bad, 4));
  MFP_CHECK(tmp.alloc((void **)&to.row, nnz * 4));
  MFP_CHECK(tmp.alloc((void **)&via.row, nnz * 4));
  MFP_CHECK(tmp.alloc((void **)&via.col, nnz * 4));
  MFP_CHECK(tmp.alloc((void **)&via.val, nnz * sizeof(V)));
  MFP_CHECK(fill_u32(bad, 0, 1, s));
  MFP_CHECK(sort_entries(tr_rows, tr_cols, tr_vals, nnz, 0, rows, rows, cols, to, via, bad, s));
  k_row_starts<<<ceil_div_u32((uint64_t)rows + 1, 256), 256, 0, s>>>(rows, nnz, to.row, row_ptr);
  MFP_HIP(hipGetLastError());
  uint32_t hbad = 0;
  MFP_HIP(hipMemcpyAsync(&hbad, bad, 4, hipMemcpyDeviceToHost, s));
  MFP_CHECK(tmp.settle(s));
  if (hbad) {
    set_error("triplet row/col index out of range");
    return MFP_ERR_ARG;
  }
  return MFP_OK;
}

// Triplets -> CSR: the sort by (row, column), ties in input order; the row
// pointers are searched in the sorted rows.
int csr_from_triplets_device(int dtype, uint32_t rows, uint32_t cols, uint64_t nnz,
                             const uint32_t *tr_rows, const uint32_t *tr_cols,
                             const double *tr_vals, uint32_t *row_ptr, uint32_t *columns,
                             void *values, hipStream_t s)
{
  MFP_ARG(nnz < (1ull << 32), "nnz must fit in 32 bits");
  if (nnz == 0) return fill_u32(row_ptr, 0, (uint64_t)rows + 1, s);
  if (dtype == MFP_F32)
    return csr_from_triplets_t(rows, cols, nnz, tr_rows, tr_cols, tr_vals, row_ptr, columns, (float *)values, s);
  return csr_from_triplets_t(rows, cols, nnz, tr_rows, tr_cols, tr_vals, row_ptr, columns, (double *)values, s);
}

// ---------------------------------------------------------------------------
// Row statistics (get_rows_statistics, common/matrix_converter.cpp:95-127).
// min/max/sum exactly; sum of squared deviations from the integer average in
// u64 (exact; equals the reference's double sum whenever that sum is below
// 2^53, where every partial double sum is exact), as sum len^2 - 2 avg sum len
// + rows avg^2 in the same modular arithmetic.  One pass: a workgroup reduces
// its rows in registers and LDS and writes one record (300,007 rows: 5 us,
// where five atomics per lane on one address took 220 + 80 us), the host adds
// the records.
// ---------------------------------------------------------------------------
struct stats_acc {
  uint32_t mn, mx;
  unsigned long long sum, sq;
};

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += (unsigned long long)__shfl_xor((long long)v, d, 64);
  return v;
}

constexpr uint32_t STATS_GRID = 512;

__global__ __launch_bounds__(256) void k_row_stats(const uint32_t *__restrict__ rp, uint32_t rows,
                                                   stats_acc *__restrict__ out)
{
  __shared__ stats_acc part[4];
  uint32_t mn = 0xFFFFFFFEu, mx = 0; // min starts at UINT_MAX-1 (:98)
  unsigned long long sum = 0, sq = 0;
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < rows; i += stride) {
    const uint32_t len = rp[i + 1] - rp[i];
    mn = min(mn, len);
    mx = max(mx, len);
    sum += len;
    sq += (unsigned long long)len * len;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    mn = min(mn, (uint32_t)__shfl_xor((int)mn, d, 64));
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, d, 64));
  }
  sum = wave_sum_u64(sum);
  sq = wave_sum_u64(sq);
  if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = stats_acc{mn, mx, sum, sq};
  __syncthreads();
  if (threadIdx.x == 0) {
    stats_acc a = part[0];
    for (int w = 1; w < 4; w++) {
      a.mn = min(a.mn, part[w].mn);
      a.mx = max(a.mx, part[w].mx);
      a.sum += part[w].sum;
      a.sq += part[w].sq;
    }
    out[blockIdx.x] = a;
  }
}

int row_stats_device(uint32_t rows, const uint32_t *rp, mfp_row_stats *out, hipStream_t s)
{
  stats_acc h{0xFFFFFFFEu, 0u, 0ull, 0ull};
  if (rows) {
    const uint32_t g = std::min<uint32_t>(ceil_div_u32(rows, 256), STATS_GRID);
    device_temps tmp;
    stats_acc *acc = nullptr;
    MFP_CHECK(tmp.alloc((void **)&acc, STATS_GRID * sizeof(stats_acc)));
    k_row_stats<<<g, 256, 0, s>>>(rp, rows, acc);
    MFP_HIP(hipGetLastError());
    std::vector<stats_acc> part(g);
    MFP_HIP(hipMemcpyAsync(part.data(), acc, g * sizeof(stats_acc), hipMemcpyDeviceToHost, s));
    MFP_CHECK(tmp.settle(s));
    for (const stats_acc &p : part) {
      h.mn = std::min(h.mn, p.mn);
      h.mx = std::max(h.mx, p.mx);
      h.sum += p.sum;
      h.sq += p.sq;
    }
  }
  const uint32_t avg = rows ? (uint32_t)h.sum / rows : 0u; // 32-bit sum as the reference
  const unsigned long long dev = h.sq - 2ull * avg * h.sum + (unsigned long long)rows * avg * avg;
  out->min_elements_in_rows = h.mn;
  out->max_elements_in_rows = h.mx;
  out->avg_elements_in_rows = avg;
  out->elements_in_rows_std_deviation = rows ? std::sqrt((double)dev / rows) : 0.0;
  return MFP_OK;
}

// ---------------------------------------------------------------------------
// ELL (common/matrix_converter.cpp:139-203): data[row + k*rows], pad (0, 0),
// rows longer than the width truncated.  Every slot is written.
// ---------------------------------------------------------------------------
// A workgroup turns 64 rows x 16 slots around in LDS: 16 lanes read a row's
// 16 entries, then 64 lanes write one slot of 64 rows (5.1M entries, width
// 64: 69 us with a lane per row reading along its own row).  Four lanes per row:
// from 2^30 rows on a launch cannot hold them all, and the workgroups go on to
// further tiles.
constexpr uint32_t ELLB_R = 64, ELLB_S = 16, ELLB_GRID = 1u << 22;

template <typename T>
__global__ __launch_bounds__(256) void k_ell_build(uint32_t rows, const uint32_t *__restrict__ rp,
                                                   const uint32_t *__restrict__ ci, const T *__restrict__ a,
                                                   uint32_t width, T *__restrict__ ev, uint32_t *__restrict__ ec)
{
  __shared__ T sv[ELLB_R][ELLB_S + 1];
  __shared__ uint32_t sc[ELLB_R][ELLB_S + 1];
  __shared__ uint32_t srp[ELLB_R + 1];
  const uint32_t t = threadIdx.x;
  for (uint64_t r0 = (uint64_t)blockIdx.x * ELLB_R; r0 < rows; r0 += (uint64_t)gridDim.x * ELLB_R) {
    if (t <= ELLB_R) srp[t] = rp[min(r0 + t, (uint64_t)rows)];
    __syncthreads();
    for (uint32_t k0 = blockIdx.y * ELLB_S; k0 < width; k0 += gridDim.y * ELLB_S) {
#pragma unroll
      for (uint32_t q = 0; q < ELLB_R * ELLB_S / 256; q++) {
        const uint32_t lr = q * (256 / ELLB_S) + t / ELLB_S, k = k0 + t % ELLB_S;
        const uint32_t s = srp[lr], len = srp[lr + 1] - s;
        const bool in = k < len;
        sv[lr][t % ELLB_S] = in ? a[s + k] : (T)0;
        sc[lr][t % ELLB_S] = in ? ci[s + k] : 0u;
      }
      __syncthreads();
#pragma unroll
      for (uint32_t q = 0; q < ELLB_R * ELLB_S / 256; q++) {
        const uint32_t lk = q * (256 / ELLB_R) + t / ELLB_R, lr = t % ELLB_R;
        if (k0 + lk < width && r0 + lr < rows) {
          const uint64_t o = r0 + lr + (uint64_t)(k0 + lk) * rows;
          ev[o] = sv[lr][lk];
          ec[o] = sc[lr][lk];
        }
      }
      __syncthreads(); // the tile and the row starts may be written again
    }
  }
}

int ell_build_device(int dtype, uint32_t rows, const uint32_t *rp, const uint32_t *ci,
                     const void *val, uint32_t width, void *ev, uint32_t *ec, hipStream_t s)
{
  if (rows == 0 || width == 0) return MFP_OK;
  const dim3 g(std::min(ceil_div_u32(rows, ELLB_R), ELLB_GRID), std::min(ceil_div_u32(width, ELLB_S), 1024u));
  if (dtype == MFP_F32)
    k_ell_build<float><<<g, 256, 0, s>>>(rows, rp, ci, (const float *)val, width, (float *)ev, ec);
  else
    k_ell_build<double><<<g, 256, 0, s>>>(rows, rp, ci, (const double *)val, width, (double *)ev, ec);
  MFP_HIP(hipGetLastError());
  return MFP_OK;
}

// ---------------------------------------------------------------------------
// COO (common/matrix_converter.cpp:211-280): CSR order, entries whose in-row
// offset is >= element_start.  Element-parallel, the rows of a tile of CSR
// elements found together.
// ---------------------------------------------------------------------------
__global__ void k_tail_counts(uint32_t rows, const uint32_t *__restrict__ rp, uint32_t e0,
                              uint32_t *__restrict__ cnt)
{
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const uint32_t len = rp[r + 1] - rp[r];
  cnt[r] = len > e0 ? len - e0 : 0u;
}

// COO entries from CSR: entry e of row r with in-row offset k >= e0 to
// position toff[r] + k - e0 (toff null: e0 = 0, position e)
template <typename T>
__global__ __launch_bounds__(ROWS_T) void k_coo_build(uint32_t rows, uint64_t nnz, const uint32_t *__restrict__ rp,
                                                      const uint32_t *__restrict__ ci, const T *__restrict__ a,
                                                      uint32_t e0, const uint32_t *__restrict__ toff,
                                                      T *__restrict__ cv, uint32_t *__restrict__ cc,
                                                      uint32_t *__restrict__ cr)
{
  __shared__ uint32_t mark[ROWS_TILE];
  __shared__ uint32_t sh[8];
  const uint32_t t0 = blockIdx.x * ROWS_TILE, t = threadIdx.x;
  const uint64_t t1 = min(nnz, (uint64_t)t0 + ROWS_TILE);
  uint32_t row[ROWS_I];
  tile_rows(rp, rows, block_row_of(rp, rows, t0, sh + 4), t0, t1, mark, sh, row);
  __syncthreads();
  // through LDS, so that neighbouring lanes handle neighbouring entries
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) mark[t * ROWS_I + k] = row[k];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) {
    const uint32_t l = k * ROWS_T + t;
    const uint64_t e = (uint64_t)t0 + l;
    if (e >= t1) break;
    const uint32_t r = mark[l];
    uint64_t o = e;
    if (toff) {
      const uint32_t in = (uint32_t)e - rp[r];
      if (in < e0) continue;
      o = toff[r] + (in - e0);
    }
    cv[o] = a[e];
    cc[o] = ci[e];
    cr[o] = r;
  }
}

int coo_tail_build_device(int dtype, uint32_t rows, uint64_t nnz, const uint32_t *rp,
                          const uint32_t *ci, const void *val, uint32_t e0, void **cv,
                          uint32_t **cc, uint32_t **cr, uint64_t *count, hipStream_t s)
{
  *cv = nullptr;
  *cc = nullptr;
  *cr = nullptr;
  device_temps tmp;
  uint32_t *toff = nullptr;
  uint32_t total = (uint32_t)nnz;
  if (e0) { // e0 = 0 takes every entry, in place
    MFP_CHECK(tmp.alloc((void **)&toff, ((uint64_t)rows + 1) * 4));
    if (rows) {
      k_tail_counts<<<ceil_div_u32(rows, 256), 256, 0, s>>>(rows, rp, e0, toff);
      MFP_HIP(hipGetLastError());
    }
    MFP_CHECK(exclusive_scan_u32(toff, toff, rows, s, &total));
  }
  *count = total;
  const size_t vs = dtype_size(dtype);
  MFP_CHECK(dmalloc(cv, (uint64_t)total * vs));
  MFP_CHECK(dmalloc((void **)cc, (uint64_t)total * 4));
  MFP_CHECK(dmalloc((void **)cr, (uint64_t)total * 4));
  if (total) {
    const uint32_t g = ceil_div_u32(nnz, ROWS_TILE);
    if (dtype == MFP_F32)
      k_coo_build<float><<<g, ROWS_T, 0, s>>>(rows, nnz, rp, ci, (const float *)val, e0, toff, (float *)*cv, *cc,
                                              *cr);
    else
      k_coo_build<double><<<g, ROWS_T, 0, s>>>(rows, nnz, rp, ci, (const double *)val, e0, toff, (double *)*cv, *cc,
                                               *cr);
    MFP_HIP(hipGetLastError());
  }
  MFP_CHECK(tmp.settle(s));
  return MFP_OK;
}

// ---------------------------------------------------------------------------
// SCOO slice pointers (common/scoo_matrix_class.cpp:74-100): slice s starts
// at row s*slice_size; entry [real slices] = nnz; the rest stay 0.
// ---------------------------------------------------------------------------
__global__ void k_scoo_slices(uint32_t rows, uint64_t nnz, const uint32_t *__restrict__ rp,
                              uint32_t slices_count, uint32_t ss, uint32_t *__restrict__ sp)
{
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > slices_count) return;
  const uint32_t real = rows ? (uint32_t)(((uint64_t)rows + ss - 1) / ss) : 0u;
  sp[s] = s < real ? rp[(uint64_t)s * ss] : (s == real ? (uint32_t)nnz : 0u);
}

int scoo_slices_device(uint32_t rows, uint64_t nnz, const uint32_t *rp, uint32_t slices_count,
                       uint32_t ss, uint32_t *sp, hipStream_t s)
{
  MFP_ARG(ss > 0, "slice_size must be positive");
  k_scoo_slices<<<ceil_div_u32((uint64_t)slices_count + 1, 256), 256, 0, s>>>(rows, nnz, rp,
                                                                             slices_count, ss, sp);
  MFP_HIP(hipGetLastError());
  return MFP_OK;
}

// ---------------------------------------------------------------------------
// Column-sorted sliced COO.  Rows longer than a threshold T ("long rows")
// are moved to their own slices, R of them per slice, in row order; every
// other row stays in the slice of R consecutive rows that holds it.  Inside a
// slice the entries are ordered by column (stable, so equal columns keep row
// order).  Each slice is cut into work items of about equal entry counts.
// When every item's column span fits in 32 - log2(R) bits, an entry stores
// one u32 (column - item base) << log2(R) | local row; otherwise a u32 column
// and a u16 local row.
// ---------------------------------------------------------------------------
__global__ void k_long_flags(uint32_t rows, const uint32_t *__restrict__ rp, uint32_t T,
                             uint32_t *__restrict__ flag)
{
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < rows) flag[r] = rp[r + 1] - rp[r] > T ? 1u : 0u;
}

__global__ void k_long_list(uint32_t rows, const uint32_t *__restrict__ flag, const uint32_t *__restrict__ rank,
                            uint32_t *__restrict__ list)
{
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < rows && flag[r]) list[rank[r]] = (uint32_t)r;
}

__global__ void k_long_mask(uint32_t rows, const uint32_t *__restrict__ flag, uint32_t *__restrict__ mask)
{
  const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
  if ((uint64_t)w * 32 >= rows) return;
  uint32_t m = 0;
  for (uint32_t b = 0; b < 32 && (uint64_t)w * 32 + b < rows; b++) m |= flag[(uint64_t)w * 32 + b] << b;
  mask[w] = m;
}

// vrow[e] = the slot of entry e's row among S R slice rows: slice R + local
// row, a long row's in the long-row slices
__global__ __launch_bounds__(ROWS_T) void k_entry_vrow(uint32_t rows, uint64_t nnz, const uint32_t *__restrict__ rp,
                                                       uint32_t long0, const uint32_t *__restrict__ mask,
                                                       const uint32_t *__restrict__ rank, uint32_t *__restrict__ vrow)
{
  __shared__ __align__(16) uint32_t mark[ROWS_TILE];
  __shared__ uint32_t sh[8];
  const uint32_t t0 = blockIdx.x * ROWS_TILE, t = threadIdx.x;
  const uint64_t t1 = min(nnz, (uint64_t)t0 + ROWS_TILE);
  uint32_t row[ROWS_I];
  tile_rows(rp, rows, block_row_of(rp, rows, t0, sh + 4), t0, t1, mark, sh, row);
  if (mask) {
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++)
      if ((mask[row[k] >> 5] >> (row[k] & 31u)) & 1u) row[k] = long0 + rank[row[k]];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) mark[t * ROWS_I + k] = row[k];
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < ROWS_I; k++) {
    const uint32_t l = k * ROWS_T + t;
    if (t0 + (uint64_t)l < t1) vrow[t0 + (uint64_t)l] = mark[l];
  }
}

// sp[s] = first sorted position whose slice is >= s
// bb[sl (nb + 1) + k] = first entry of slice sl whose column is >= k W
// (entries of a slice are sorted by column), for k = 0..nb
__global__ void k_band_bounds(uint32_t S, uint32_t nb, uint64_t W, const uint32_t *__restrict__ sp,
                              const uint32_t *__restrict__ col_sorted, uint32_t *__restrict__ bb)
{
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint64_t)S * (nb + 1)) return;
  const uint32_t sl = (uint32_t)(t / (nb + 1)), k = (uint32_t)(t % (nb + 1));
  uint32_t lo = sp[sl], hi = sp[sl + 1];
  const uint64_t c0 = (uint64_t)k * W;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if ((uint64_t)col_sorted[mid] < c0)
      lo = mid + 1;
    else
      hi = mid;
  }
  bb[t] = lo;
}

__global__ void k_slice_bounds(uint32_t S, uint64_t nnz, const uint32_t *__restrict__ vrow_sorted, uint32_t rbits,
                               uint32_t *__restrict__ sp)
{
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > S) return;
  uint64_t lo = 0, hi = nnz;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) / 2;
    if ((vrow_sorted[mid] >> rbits) < s)
      lo = mid + 1;
    else
      hi = mid;
  }
  sp[s] = (uint32_t)lo;
}

// Column span of each slice: last column - first column of its sorted entries.
__global__ void k_slice_span(uint32_t S, const uint32_t *__restrict__ sp, const uint32_t *__restrict__ col_sorted,
                             uint32_t *__restrict__ span)
{
  const uint32_t sl = blockIdx.x * blockDim.x + threadIdx.x;
  if (sl >= S) return;
  const uint32_t lo = sp[sl], hi = sp[sl + 1];
  span[sl] = hi > lo ? col_sorted[hi - 1] - col_sorted[lo] : 0u;
}

__global__ void k_item_base(uint32_t NI, const uint4 *__restrict__ items, const uint32_t *__restrict__ col,
                            uint32_t *__restrict__ base, uint32_t *__restrict__ max_span)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NI) return;
  const uint32_t e0 = items[i].y, e1 = items[i].z;
  if (e1 > e0) {
    base[i] = col[e0];
    atomicMax(max_span, col[e1 - 1] - col[e0]);
  } else {
    base[i] = 0;
  }
}

// Sorted entries to their words.  A workgroup takes 1024 positions, in order;
// the item holding its first one is searched once, later ones by advancing.
template <typename T>
__global__ __launch_bounds__(256) void k_cs_place(uint64_t nnz, const uint32_t *__restrict__ vrow,
                                                  const uint32_t *__restrict__ col, const T *__restrict__ a, uint32_t NI,
                                                  const uint4 *__restrict__ items, const uint32_t *__restrict__ base,
                                                  uint32_t rbits, T *__restrict__ ev, uint32_t *__restrict__ ec)
{
  const uint64_t p0 = (uint64_t)blockIdx.x * 1024u;
  // the last item with e0 <= p0 (items are in position order and cover every
  // position; of empty items at one position the last comes out, and the
  // position then belongs to it or to a later one)
  uint32_t lo = 0, hi = NI;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (items[mid].y <= p0)
      lo = mid;
    else
      hi = mid;
  }
  uint32_t e0 = items[lo].y, e1 = items[lo].z;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    const uint64_t i = p0 + k * 256u + threadIdx.x;
    if (i >= nnz) return;
    while (i >= e1) {
      lo++;
      e0 = items[lo].y;
      e1 = items[lo].z;
    }
    const uint32_t c = col[i], w = ((c - base[lo]) << rbits) | (vrow[i] & ((1u << rbits) - 1u));
    // inside an aligned block of 256 positions that lies wholly in one
    // item, position 64 j + l goes to word l, slot j: lane l's 16-byte word
    // then holds the block's positions l, 64 + l, 128 + l and 192 + l, so
    // each of the wave's four gathers reads 64 consecutive columns
    const uint64_t b0 = i & ~(uint64_t)255;
    const bool in_block = b0 >= e0 && b0 + 256 <= e1;
    const uint64_t d = in_block ? b0 + 4 * (i & 63) + ((i >> 6) & 3) : i;
    // FP64 values of such a block: slots 0 and 1 of its 64 words first, as
    // 64 consecutive 16-byte pairs, then slots 2 and 3, so that each 16-byte
    // value load of a wave reads 1 KiB contiguous
    const uint64_t dv = sizeof(T) == 8 && in_block ? b0 + (((i >> 7) & 1) << 7) + 2 * (i & 63) + ((i >> 6) & 1) : d;
    ev[dv] = a[i];
    ec[d] = w;
  }
}

// Entries of the CSR matrix sorted by (slice, column), stably: vrow, columns
// and values into `to`.
template <typename T>
static int cs_sort_t(uint32_t rows, uint32_t cols, uint64_t nnz, const uint32_t *rp, const uint32_t *ci, const void *val,
                     uint32_t rbits, uint32_t S_reg, uint32_t S, const uint32_t *mask, const uint32_t *rank,
                     const sort_arrays<T> &to, const sort_arrays<T> &via, hipStream_t s)
{
  // the first pass reads the rows from the side that it does not write
  const uint32_t bits = (cols ? bit_length(cols - 1) : 0) + (S ? bit_length(S - 1) : 0);
  uint32_t *vrow = std::max(1u, (bits + 7) / 8) % 2 ? via.row : to.row;
  k_entry_vrow<<<ceil_div_u32(nnz, ROWS_TILE), ROWS_T, 0, s>>>(rows, nnz, rp, S_reg << rbits, mask, rank, vrow);
  MFP_HIP(hipGetLastError());
  return sort_entries(vrow, ci, (const T *)val, nnz, rbits, S, 0, cols, to, via, nullptr, s);
}

template <typename T>
static int cs_place_t(uint64_t nnz, const void *sorted_row, const void *sorted_col, const void *sorted_val, uint32_t NI,
                      const uint4 *items, const uint32_t *base, uint32_t rbits, void *ev, uint32_t *ec, hipStream_t s)
{
  k_cs_place<T><<<ceil_div_u32(nnz, 1024), 256, 0, s>>>(nnz, (const uint32_t *)sorted_row, (const uint32_t *)sorted_col,
                                                        (const T *)sorted_val, NI, items, base, rbits, (T *)ev, ec);
  MFP_HIP(hipGetLastError());
  return MFP_OK;
}

int scoo_cs_build_device(int dtype, uint32_t rows, uint32_t cols, uint64_t nnz, const uint32_t *rp,
                         const uint32_t *ci, const void *val, uint32_t R, uint32_t long_threshold,
                         uint64_t item_entries, scoo_cs_layout *out, hipStream_t s,
                         bool own_partials)
{
  MFP_ARG(R >= 1 && R <= 65536 && (R & (R - 1)) == 0,
          "column-sorted SCOO slice size must be a power of two <= 65536");
  MFP_ARG(nnz < (1ull << 32), "nnz must fit in 32 bits");
  MFP_ARG(item_entries >= 1, "entries per work item must be positive");
  *out = scoo_cs_layout{};
  uint32_t rbits = 0;
  while ((1u << rbits) < R) rbits++;
  out->R = R;
  out->rbits = rbits;
  const uint32_t S_reg = rows ? (uint32_t)(((uint64_t)rows + R - 1) / R) : 0u;
  out->S_reg = S_reg;
  const size_t vs = dtype_size(dtype);
  std::vector<void *> tmp;
  auto scratch = [&](void **p, uint64_t bytes) {
    const int st = dmalloc(p, std::max<uint64_t>(bytes, 4));
    if (st == MFP_OK) tmp.push_back(*p);
    return st;
  };
  auto done = [&](int st) {
    const free_scope scope;
    for (void *p : tmp) dfree(p);
    if (st != MFP_OK) scoo_cs_free(out);
    return st;
  };
  int st = MFP_OK;
  // long rows: flag, rank (exclusive scan) and list
  uint32_t *flag = nullptr, *rank = nullptr;
  uint32_t NL = 0;
  if (rows && long_threshold != 0xFFFFFFFFu) {
    st = scratch((void **)&flag, (uint64_t)rows * 4);
    if (st == MFP_OK) st = scratch((void **)&rank, (uint64_t)rows * 4);
    if (st != MFP_OK) return done(st);
    k_long_flags<<<ceil_div_u32(rows, 256), 256, 0, s>>>(rows, rp, long_threshold, flag);
    if (hipGetLastError() != hipSuccess) return done(MFP_ERR_HIP);
    st = exclusive_scan_u32(flag, rank, rows, s, &NL);
    if (st != MFP_OK) return done(st);
  }
  // the rows of all slices are numbered in 32 bits
  if (((uint64_t)S_reg + ((uint64_t)NL + R - 1) / R) << rbits > 1ull << 32) NL = 0;
  out->NL = NL;
  out->S_long = (uint32_t)(((uint64_t)NL + R - 1) / R);
  const uint32_t S = S_reg + out->S_long;
  out->S = S;
  st = dmalloc((void **)&out->long_rows, std::max<uint64_t>(NL, 1) * 4);
  if (st == MFP_OK) st = dmalloc((void **)&out->sp, ((uint64_t)S + 1) * 4);
  if (st == MFP_OK && NL) st = dmalloc((void **)&out->long_mask, ((uint64_t)rows + 31) / 32 * 4);
  if (st != MFP_OK) return done(st);
  if (NL) {
    k_long_list<<<ceil_div_u32(rows, 256), 256, 0, s>>>(rows, flag, rank, out->long_rows);
    k_long_mask<<<ceil_div_u32(((uint64_t)rows + 31) / 32, 256), 256, 0, s>>>(rows, flag, out->long_mask);
    if (hipGetLastError() != hipSuccess) return done(MFP_ERR_HIP);
  }
  // the entries sorted by (slice, column), through the plan's own arrays
  st = dmalloc(&out->ev, std::max<uint64_t>(nnz, 1) * vs);
  if (st == MFP_OK) st = dmalloc((void **)&out->ec, std::max<uint64_t>(nnz, 1) * 4);
  uint32_t *span = nullptr, *srow = nullptr, *scol = nullptr, *vrow = nullptr;
  void *sval = nullptr;
  if (st == MFP_OK) st = scratch((void **)&span, 4);
  if (st == MFP_OK) st = scratch((void **)&srow, nnz * 4);
  if (st == MFP_OK) st = scratch((void **)&scol, nnz * 4);
  if (st == MFP_OK) st = scratch(&sval, nnz * vs);
  if (st == MFP_OK) st = scratch((void **)&vrow, nnz * 4);
  if (st != MFP_OK) return done(st);
  if (nnz) {
    auto sort = [&](auto tv) {
      using T = decltype(tv);
      return cs_sort_t<T>(rows, cols, nnz, rp, ci, val, rbits, S_reg, S, NL ? out->long_mask : nullptr, rank,
                          sort_arrays<T>{srow, scol, (T *)sval}, sort_arrays<T>{vrow, out->ec, (T *)out->ev}, s);
    };
    st = vs == 2 ? sort(uint16_t()) : vs == 4 ? sort(uint32_t()) : sort(uint64_t());
    if (st != MFP_OK) return done(st);
  }
  // slice boundaries, then work items on the host
  k_slice_bounds<<<ceil_div_u32((uint64_t)S + 1, 256), 256, 0, s>>>(S, nnz, srow, rbits, out->sp);
  if (hipGetLastError() != hipSuccess) return done(MFP_ERR_HIP);
  std::vector<uint32_t> hsp((size_t)S + 1);
  if (hipMemcpyAsync(hsp.data(), out->sp, hsp.size() * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return done(MFP_ERR_HIP);
  // Column bands of width W = 2^(32 - rbits): an item whose columns span
  // less than W packs (column - item base) and the local row into one u32.
  // A slice whose columns span less than W is one band; any other slice is
  // cut at the multiples of W.  Each non-empty band of a slice is cut into
  // about E_band / item_entries equal pieces.
  const uint64_t W = rbits ? (1ull << (32 - rbits)) : (1ull << 32);
  const uint32_t nb = (uint32_t)std::max<uint64_t>(1, ((uint64_t)cols + W - 1) / W);
  std::vector<uint32_t> hbb((size_t)S * (nb + 1));
  std::vector<uint32_t> slice_span(S, 0u);
  if (S && nb > 1) {
    uint32_t *bb = nullptr, *sspan = nullptr;
    st = scratch((void **)&bb, hbb.size() * 4);
    if (st == MFP_OK) st = scratch((void **)&sspan, (uint64_t)S * 4);
    if (st != MFP_OK) return done(st);
    k_band_bounds<<<ceil_div_u32(hbb.size(), 256), 256, 0, s>>>(S, nb, W, out->sp, scol, bb);
    if (hipGetLastError() != hipSuccess) return done(MFP_ERR_HIP);
    k_slice_span<<<ceil_div_u32(S, 256), 256, 0, s>>>(S, out->sp, scol, sspan);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(hbb.data(), bb, hbb.size() * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipMemcpyAsync(slice_span.data(), sspan, (size_t)S * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return done(MFP_ERR_HIP);
    for (uint32_t sl = 0; sl < S; sl++) {
      if (slice_span[sl] >= W) continue;
      uint32_t *b = &hbb[(size_t)sl * (nb + 1)];
      b[0] = hsp[sl]; // the whole slice in band 0, the other bands empty
      for (uint32_t k = 1; k <= nb; k++) b[k] = hsp[sl + 1];
    }
  } else {
    for (uint32_t sl = 0; sl < S; sl++) {
      hbb[(size_t)sl * 2] = hsp[sl];
      hbb[(size_t)sl * 2 + 1] = hsp[sl + 1];
    }
  }
  std::vector<uint4> items;
  std::vector<uint4> fin, finl; // finish blocks {slice, first partial slot, slots, first row in the slice}
  uint32_t slots = 0;
  std::vector<std::pair<uint32_t, uint32_t>> cuts; // [e0, e1) of the slice's items
  for (uint32_t sl = 0; sl < S; sl++) {
    cuts.clear();
    for (uint32_t k = 0; k < nb; k++) {
      const uint32_t b0 = hbb[(size_t)sl * (nb + 1) + k], b1 = hbb[(size_t)sl * (nb + 1) + k + 1];
      const uint64_t Eb = b1 - b0;
      if (Eb == 0) continue;
      const uint64_t nk = std::max<uint64_t>(1, (Eb + item_entries / 2) / item_entries);
      for (uint64_t q = 0; q < nk; q++)
        cuts.push_back({b0 + (uint32_t)(Eb * q / nk), b0 + (uint32_t)(Eb * (q + 1) / nk)});
    }
    if (cuts.empty()) cuts.push_back({hsp[sl], hsp[sl]}); // an empty slice still writes its zeros
    const uint32_t n = (uint32_t)cuts.size();
    // a slice with one item writes y; with several, each item fills a
    // partial slot and finish blocks add the slots in slot order
    const uint32_t mode = n == 1 ? CS_DIRECT : slots;
    if (n > 1 && sl < S_reg) {
      const uint32_t lim = (uint32_t)std::min<uint64_t>(R, (uint64_t)rows - (uint64_t)sl * R);
      for (uint32_t r0 = 0; r0 < lim; r0 += 4 * CS_FIN_ROWS) fin.push_back(make_uint4(sl, slots, n, r0));
    } else if (n > 1) {
      // a long-row slice can have many items: a wave per row adds its slots
      const uint32_t lim = (uint32_t)std::min<uint64_t>(R, (uint64_t)NL - (uint64_t)(sl - S_reg) * R);
      for (uint32_t r0 = 0; r0 < lim; r0 += CS_FIN_LONG) finl.push_back(make_uint4(sl, slots, n, r0));
    }
    for (uint32_t k = 0; k < n; k++)
      items.push_back(make_uint4(sl, cuts[k].first, cuts[k].second, mode < CS_DIRECT ? mode + k : mode));
    if (mode < CS_DIRECT) slots += n;
  }
  out->NFR = (uint32_t)fin.size();
  fin.insert(fin.end(), finl.begin(), finl.end());
  out->NI = (uint32_t)items.size();
  out->NF = (uint32_t)fin.size();
  out->slots = slots;
  st = dmalloc((void **)&out->items, std::max<size_t>(items.size(), 1) * sizeof(uint4));
  if (st == MFP_OK) st = dmalloc((void **)&out->fin, std::max<size_t>(fin.size(), 1) * sizeof(uint4));
  if (st == MFP_OK) st = dmalloc((void **)&out->base, std::max<size_t>(items.size(), 1) * 4);
  // partial slots hold the vector type: float for FP32 and 16-bit values;
  // FP32 / FP64 plans also serve SpMM with k columns while R k doubles fit
  // in LDS, so their slots hold kmax columns
  const size_t ps = dtype == MFP_F64 ? 8 : 4;
  out->kmax = 1;
  if (dtype == MFP_F32 || dtype == MFP_F64)
    while (out->kmax < 16 && (uint64_t)R * out->kmax * 2 * 8 <= 163840) out->kmax *= 2;
  if (st == MFP_OK && slots && own_partials) st = dmalloc(&out->partial, (uint64_t)slots * R * out->kmax * ps);
  if (st != MFP_OK) return done(st);
  if (!items.empty() &&
      hipMemcpyAsync(out->items, items.data(), items.size() * sizeof(uint4), hipMemcpyHostToDevice, s) != hipSuccess)
    return done(MFP_ERR_HIP);
  if (!fin.empty() &&
      hipMemcpyAsync(out->fin, fin.data(), fin.size() * sizeof(uint4), hipMemcpyHostToDevice, s) != hipSuccess)
    return done(MFP_ERR_HIP);
  st = fill_u32(span, 0, 1, s);
  if (st != MFP_OK) return done(st);
  if (out->NI) {
    k_item_base<<<ceil_div_u32(out->NI, 256), 256, 0, s>>>(out->NI, out->items, scol, out->base, span);
    if (hipGetLastError() != hipSuccess) return done(MFP_ERR_HIP);
  }
  uint32_t hspan = 0;
  if (hipMemcpyAsync(&hspan, span, 4, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
    return done(MFP_ERR_HIP);
  // every item lies inside one column band, so its offsets fit beside the row
  if (rbits && (uint64_t)hspan >= (1ull << (32 - rbits))) {
    set_error("column-sorted SCOO: an item spans more than its column band");
    return done(MFP_ERR_STATE);
  }
  if (nnz) {
    st = (vs == 2 ? cs_place_t<uint16_t> : vs == 4 ? cs_place_t<uint32_t> : cs_place_t<uint64_t>)(
        nnz, srow, scol, sval, out->NI, out->items, out->base, rbits, out->ev, out->ec, s);
    if (st != MFP_OK) return done(st);
  }
  if (hipStreamSynchronize(s) != hipSuccess) {
    set_error("column-sorted SCOO build failed");
    return done(MFP_ERR_HIP);
  }
  // Launch order: piece k of n covers about columns [k/n, (k+1)/n) of its
  // slice, so ordering the items by the centre of that band (then by slice)
  // gives each XCD's contiguous range of items one band of x for its L2.
  // The placement above needed the items in entry order; the kernel does not.
  if (out->NI > 1) {
    std::vector<uint32_t> hbase(out->NI);
    if (hipMemcpyAsync(hbase.data(), out->base, (size_t)out->NI * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return done(MFP_ERR_HIP);
    std::vector<uint32_t> pieces(out->NI), order(out->NI);
    for (uint32_t i = 0; i < out->NI;) { // items of one slice are adjacent
      uint32_t j = i;
      while (j < out->NI && items[j].x == items[i].x) j++;
      for (uint32_t k = i; k < j; k++) pieces[k] = j - i;
      i = j;
    }
    std::vector<uint32_t> first(out->NI);
    for (uint32_t i = 0; i < out->NI; i++) first[i] = (i && items[i - 1].x == items[i].x) ? first[i - 1] : i;
    for (uint32_t i = 0; i < out->NI; i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
      // band centre (2k + 1) / (2n), compared exactly as a cross product
      const uint64_t ka = a - first[a], kb = b - first[b];
      return (2 * ka + 1) * pieces[b] < (2 * kb + 1) * pieces[a];
    });
    // The kernel maps workgroups to items with xcd_block: XCD x runs one
    // contiguous range of this order, first those of its items that fill its
    // CUs, then the rest as CUs free up.  Items of ordinary slices take about
    // twice as long as long-row items, so each range gets an even share of
    // them, placed first, then long-row items (both in band-centre order, so
    // each XCD still works on one band of x).  Left to the band-centre order
    // alone, one XCD can receive more ordinary items than it has CUs and run
    // two of them back to back while others idle.
    if (out->NI >= 32) {
      std::vector<uint32_t> ro, lo;
      for (uint32_t i : order) (items[i].x < S_reg ? ro : lo).push_back(i);
      const uint32_t nr = (uint32_t)ro.size(), nl = (uint32_t)lo.size();
      const uint32_t q = out->NI / 8, rem = out->NI % 8;
      uint32_t ri = 0, li = 0, p0 = 0;
      for (uint32_t x = 0; x < 8; x++) {
        const uint32_t len = q + (x < rem ? 1u : 0u);
        const uint32_t share = (uint32_t)((uint64_t)nr * (x + 1) / 8 - (uint64_t)nr * x / 8);
        uint32_t rx = std::min({share, len, nr - ri});
        const uint32_t lx = std::min(len - rx, nl - li);
        rx += std::min(len - rx - lx, nr - ri - rx); // no long-row items left: more ordinary ones
        for (uint32_t k = 0; k < rx; k++) order[p0++] = ro[ri++];
        for (uint32_t k = 0; k < lx; k++) order[p0++] = lo[li++];
      }
      // every range is filled exactly: the ranges' lengths add up to NI
      if (p0 != out->NI || ri != nr || li != nl) {
        set_error("column-sorted SCOO: work item ordering failed");
        return done(MFP_ERR_STATE);
      }
    }
    std::vector<uint4> it2(out->NI);
    std::vector<uint32_t> b2(out->NI);
    for (uint32_t i = 0; i < out->NI; i++) {
      it2[i] = items[order[i]];
      b2[i] = hbase[order[i]];
    }
    if (hipMemcpyAsync(out->items, it2.data(), it2.size() * sizeof(uint4), hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(out->base, b2.data(), b2.size() * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return done(MFP_ERR_HIP);
  }
  out->device_bytes = nnz * (vs + 4) + ((uint64_t)S + 1) * 4 +
                      (uint64_t)out->NI * 20 + (uint64_t)out->NF * 16 + (uint64_t)NL * 4 +
                      (NL ? ((uint64_t)rows + 31) / 32 * 4 : 0) +
                      (own_partials ? (uint64_t)slots * R * out->kmax * ps : 0);
  return done(MFP_OK);
}

void scoo_cs_free(scoo_cs_layout *l)
{
  const free_scope scope;
  dfree(l->sp);
  dfree(l->long_rows);
  dfree(l->long_mask);
  dfree(l->items);
  dfree(l->fin);
  dfree(l->base);
  dfree(l->partial);
  dfree(l->ev);
  dfree(l->ec);
  *l = scoo_cs_layout{};
}

// ---------------------------------------------------------------------------
// Row blocks (fill_row_blocks, gpu/csr_adaptive_spmv.cu:180-240) in parallel.
// The greedy partition is a chain 0 -> close(0) -> ...: close(s) is the row
// where a block started at s closes (or NONE when the loop ends first), and it
// depends on s only.  The chain's nodes in [0, rows] in order, followed by rows,
// are the reference's output.
//   k_close      close(s) of every row, by binary search in the row pointers
//                (they only grow, so the first row that fills the block can be
//                searched)
//   k_seg_exit   a segment of SEG nodes finds, by pointer jumping in LDS,
//                where a chain from each node leaves the segment
//   k_seg_chase  one lane follows the chain from segment to segment
//   k_seg_mark   each segment marks the chain from its entry node, in LDS
//   k_seg_write  the marked nodes in order
// Jumping over all nodes in HBM took two launches per doubling, 40 and more
// in all, and close(s) up to W serial steps per node.
// ---------------------------------------------------------------------------
// Segments of 16,384 rows, of 4,096 up to 262,144 rows (more workgroups, and
// at most 64 steps of the chase).
constexpr uint32_t SEG_T = 1024;
constexpr uint32_t NO_NODE = 0xFFFFFFFFu;

// close(s) for s < rows, always above s; rows also where the loop ends first
__device__ __forceinline__ uint32_t close_of(uint32_t s, uint32_t rows, const uint32_t *__restrict__ rp, uint32_t W)
{
  const uint32_t b = rp[s];
  const uint64_t end = min((uint64_t)rows, (uint64_t)s + W + 1u);
  uint64_t lo = s, hi = end + 1; // rp[lo] - b < W; hi: first row known to reach W, or end + 1
  while (hi - lo > 1) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if (rp[mid] - b >= W)
      hi = mid;
    else
      lo = mid;
  }
  // full at row hi: closes there when exactly full or when it holds one row,
  // else before it; not full: closes at end, after W + 1 rows or with the matrix
  if (hi <= end) return (uint32_t)(rp[hi] - b == W || hi - s == 1 ? hi : hi - 1);
  return (uint32_t)end;
}

__global__ __launch_bounds__(256) void k_close(uint32_t rows, const uint32_t *__restrict__ rp, uint32_t W,
                                               uint32_t *__restrict__ J)
{
  const uint64_t s = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (s < rows) J[s] = close_of((uint32_t)s, rows, rp, W);
}

// exit[s] = first node of s's chain outside its segment
template <uint32_t SEG>
__global__ __launch_bounds__(SEG_T) void k_seg_exit(uint32_t rows, const uint32_t *__restrict__ J,
                                                    uint32_t *__restrict__ exit, uint32_t *__restrict__ entry)
{
  constexpr uint32_t SEG_I = SEG / SEG_T;
  extern __shared__ uint32_t nxt[]; // SEG
  const uint32_t s0 = blockIdx.x * SEG, n = min(SEG, rows - s0), t = threadIdx.x;
  uint32_t v[SEG_I];
#pragma unroll
  for (uint32_t k = 0; k < SEG_I; k++) {
    const uint32_t l = k * SEG_T + t;
    v[k] = l < n ? J[s0 + l] : NO_NODE;
    nxt[l] = v[k];
  }
  if (t == 0) entry[blockIdx.x] = NO_NODE;
  for (;;) {
    __syncthreads();
    bool moved = false;
#pragma unroll
    for (uint32_t k = 0; k < SEG_I; k++)
      if (v[k] - s0 < n) { // still inside (nodes only grow)
        v[k] = nxt[v[k] - s0];
        moved = true;
      }
    if (!__syncthreads_or(moved)) break;
#pragma unroll
    for (uint32_t k = 0; k < SEG_I; k++) nxt[k * SEG_T + t] = v[k];
  }
#pragma unroll
  for (uint32_t k = 0; k < SEG_I; k++) {
    const uint32_t l = k * SEG_T + t;
    if (l < n) exit[s0 + l] = v[k];
  }
}

// entry[segment] = the chain's first node in it
__global__ void k_seg_chase(uint32_t rows, uint32_t seg, const uint32_t *__restrict__ exit, uint32_t *__restrict__ entry)
{
  uint32_t node = 0;
  while (node < rows) {
    entry[node / seg] = node;
    node = exit[node]; // a later segment's, or rows
  }
}

// bits of the segment's chain nodes (SEG / 32 words per segment) and
// their count; the chain's last node says whether its block closes at rows
// (*at_end: node rows is marked too) or the loop ended first
template <uint32_t SEG>
__global__ __launch_bounds__(SEG_T) void k_seg_mark(uint32_t rows, const uint32_t *__restrict__ rp, uint32_t W,
                                                    const uint32_t *__restrict__ J,
                                                    const uint32_t *__restrict__ entry, uint32_t *__restrict__ bits,
                                                    uint32_t *__restrict__ count, uint32_t *__restrict__ at_end)
{
  constexpr uint32_t SEG_I = SEG / SEG_T;
  extern __shared__ uint32_t nxt[]; // SEG, then SEG / 32 words of marks
  uint32_t *mark = nxt + SEG;
  __shared__ uint32_t sh[SEG_T / 64];
  const uint32_t s0 = blockIdx.x * SEG, n = min(SEG, rows - s0), t = threadIdx.x;
  const uint32_t e = entry[blockIdx.x];
  static_assert(SEG / 32 <= SEG_T, "one word of marks per lane");
  uint32_t v[SEG_I];
#pragma unroll
  for (uint32_t k = 0; k < SEG_I; k++) {
    const uint32_t l = k * SEG_T + t;
    v[k] = l < n ? J[s0 + l] : NO_NODE;
    nxt[l] = v[k];
  }
  if (t < SEG / 32) mark[t] = e != NO_NODE && (e - s0) / 32 == t ? 1u << ((e - s0) & 31u) : 0u;
  if (e != NO_NODE) { // uniform
    for (;;) {
      __syncthreads();
      bool moved = false;
      // v = 2^k steps from each node: a marked node marks the one it leads to
#pragma unroll
      for (uint32_t k = 0; k < SEG_I; k++) {
        const uint32_t l = k * SEG_T + t, to = v[k] - s0;
        if (to < n) {
          if ((mark[l / 32] >> (l & 31u)) & 1u) atomicOr(&mark[to / 32], 1u << (to & 31u));
          v[k] = nxt[to];
          moved = true;
        }
      }
      if (!__syncthreads_or(moved)) break;
#pragma unroll
      for (uint32_t k = 0; k < SEG_I; k++) nxt[k * SEG_T + t] = v[k];
    }
  }
  __syncthreads();
  const uint32_t w = t < SEG / 32 ? mark[t] : 0u;
  if (t < SEG / 32) bits[(uint64_t)blockIdx.x * (SEG / 32) + t] = w;
#pragma unroll
  for (uint32_t k = 0; k < SEG_I; k++) {
    const uint32_t l = k * SEG_T + t;
    if (l < n && ((mark[l / 32] >> (l & 31u)) & 1u) && J[s0 + l] == rows) // one lane of the grid
      *at_end = rp[rows] - rp[s0 + l] >= W || (uint64_t)rows == (uint64_t)s0 + l + W + 1u ? 1u : 0u;
  }
  uint32_t total;
  (void)block_exclusive_scan<SEG_T>((uint32_t)__popc(w), sh, &total);
  if (t == 0) count[blockIdx.x] = total;
}

// the marked nodes from offs[segment] on; the first workgroup adds node rows
// when marked, and the closing rows
template <uint32_t SEG>
__global__ __launch_bounds__(SEG / 32) void k_seg_write(uint32_t rows, uint32_t nseg,
                                                             const uint32_t *__restrict__ bits,
                                                             const uint32_t *__restrict__ offs,
                                                             const uint32_t *__restrict__ at_end,
                                                             uint32_t *__restrict__ out)
{
  __shared__ uint32_t sh[SEG / 32 / 64];
  uint32_t w = bits[(uint64_t)blockIdx.x * (SEG / 32) + threadIdx.x];
  uint32_t o = offs[blockIdx.x] + block_exclusive_scan<SEG / 32>((uint32_t)__popc(w), sh, nullptr);
  uint32_t node = blockIdx.x * SEG + threadIdx.x * 32u;
  while (w) {
    const uint32_t b = (uint32_t)__ffs((int)w) - 1u;
    out[o++] = node + b;
    w &= w - 1u;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const uint32_t total = offs[nseg];
    out[total] = rows;
    if (*at_end) out[total + 1] = rows;
  }
}

template <uint32_t SEG>
static int row_blocks_t(uint32_t rows, const uint32_t *rp, uint32_t W, uint32_t **blocks_out, uint32_t *count_out,
                        hipStream_t s)
{
  device_temps tmp;
  uint32_t *out = nullptr;
  const uint32_t nseg = ceil_div_u32(rows, SEG);
  uint32_t *J = nullptr, *exit = nullptr, *entry = nullptr, *bits = nullptr, *count = nullptr;
  MFP_CHECK(tmp.alloc((void **)&J, (uint64_t)rows * 4));
  MFP_CHECK(tmp.alloc((void **)&exit, (uint64_t)rows * 4));
  MFP_CHECK(tmp.alloc((void **)&entry, (uint64_t)nseg * 4));
  MFP_CHECK(tmp.alloc((void **)&bits, (uint64_t)nseg * (SEG / 32) * 4));
  MFP_CHECK(tmp.alloc((void **)&count, ((uint64_t)nseg + 2) * 4)); // + total, at_end
  const uint32_t lds = SEG * 4, lds_mark = lds + SEG / 32 * 4;
  MFP_HIP(hipFuncSetAttribute((const void *)k_seg_exit<SEG>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  MFP_HIP(hipFuncSetAttribute((const void *)k_seg_mark<SEG>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_mark));
  k_close<<<ceil_div_u32(rows, 256), 256, 0, s>>>(rows, rp, W, J);
  k_seg_exit<SEG><<<nseg, SEG_T, lds, s>>>(rows, J, exit, entry);
  k_seg_chase<<<1, 1, 0, s>>>(rows, SEG, exit, entry);
  k_seg_mark<SEG><<<nseg, SEG_T, lds_mark, s>>>(rows, rp, W, J, entry, bits, count, count + nseg + 1);
  k_scan_offsets<<<1, 1024, 0, s>>>(count, nseg);
  MFP_HIP(hipGetLastError());
  uint32_t h[2] = {0, 0};
  MFP_HIP(hipMemcpyAsync(h, count + nseg, 8, hipMemcpyDeviceToHost, s));
  MFP_CHECK(tmp.settle(s));
  const uint32_t total = h[0] + h[1];
  MFP_CHECK(tmp.alloc((void **)&out, ((uint64_t)total + 1) * 4));
  k_seg_write<SEG><<<nseg, SEG / 32, 0, s>>>(rows, nseg, bits, count, count + nseg + 1, out);
  MFP_HIP(hipGetLastError());
  MFP_CHECK(tmp.settle(s));
  tmp.release(out);
  *blocks_out = out;
  *count_out = total;
  return MFP_OK;
}

int row_blocks_device(uint32_t rows, const uint32_t *rp, uint32_t W, uint32_t **blocks_out,
                      uint32_t *count_out, hipStream_t s)
{
  MFP_ARG(W > 0, "nnz_per_wg must be positive");
  if (rows == 0) { // node 0 is node rows: one marked node, then the closing rows
    device_temps tmp;
    uint32_t *out = nullptr;
    MFP_CHECK(tmp.alloc((void **)&out, 2 * 4));
    MFP_CHECK(fill_u32(out, 0, 2, s));
    MFP_HIP(hipStreamSynchronize(s));
    tmp.release(out);
    *blocks_out = out;
    *count_out = 1;
    return MFP_OK;
  }
  return rows > (1u << 18) ? row_blocks_t<16384>(rows, rp, W, blocks_out, count_out, s)
                           : row_blocks_t<4096>(rows, rp, W, blocks_out, count_out, s);
}

} // namespace mfp
