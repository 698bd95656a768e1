// 64-d structure features of a device CSR matrix, the format selector's input.
// Two passes accumulate integer counters (so the result does not depend on
// atomic order); the host turns them into the feature vector in double.
//
//  0 log2(rows+1)/32          1 log2(cols+1)/32         2 log2(nnz+1)/40
//  3 log2(1+mean)/16          4 log2(1+max)/16          5 min(cv, 32)/32
//  6 empty-row fraction       7 log2(1+std)/16
//  8..31  row fraction per row-length bin: 0 for empty rows, 1 + floor(log2 len)
//         capped at 23
// 32..47  nnz fraction per bin floor(log2 len) capped at 15
// 48..55  nnz fraction per relative distance d = |c rows - r cols| / (rows cols)
//         from the scaled diagonal: d < 1e-4 4^k for k = 0..6, then d >= 0.4096
// 56 mean d (d quantised down to 2^-24)   57 fraction of entries with c == r
// 58 mean over non-empty rows of (last column - first column + 1) / cols
// 59 log2(rows max / nnz)/16 (ELL padding factor, 0 when nnz = 0)
// 60 nnz fraction in rows longer than 4096   61 nnz fraction in rows of <= 4
// 62 fraction of rows longer than 64         63 constant 1
// mean, std and cv are of the row length (population std).
#include "entry_rows.h"
#include "mfp_internal.h"
#include "objects.h"
#include "wave64.h"

#include <algorithm>
#include <cmath>

namespace mfp {

// what the rows and the entries add up to; every field a u64
struct feat_row_counters {
  unsigned long long len_hist[24];
  unsigned long long nnz_hist[16];
  unsigned long long sumsq, empty, nnz_big, nnz_small, rows_gt64, span_sum, nonempty;
  unsigned long long max_len; // the one maximum, last
};
struct feat_entry_counters {
  unsigned long long dist_hist[8];
  unsigned long long dist_sum, diag;
};
constexpr int FEAT_R = sizeof(feat_row_counters) / 8, FEAT_E = sizeof(feat_entry_counters) / 8;

__device__ __forceinline__ int ilog2(uint32_t v) { return 31 - __clz(v); }

// sum over the wave's 64 lanes, in lane 0, in pieces of at most 24 bits that
// the 32-bit lane moves can add without overflow
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v)
{
  const uint32_t a = group_reduce<64>((uint32_t)(v & 0xFFFFFFu)), b = group_reduce<64>((uint32_t)(v >> 24) & 0xFFFFFFu),
                 c = group_reduce<64>((uint32_t)(v >> 48));
  return a + ((unsigned long long)b << 24) + ((unsigned long long)c << 48);
}

// the workgroup's sums of v[0..N) over 256 lanes to out[0..N); sh: 4 N words
template <int N>
__device__ __forceinline__ void block_sums(const unsigned long long (&v)[N], unsigned long long *sh,
                                           unsigned long long *__restrict__ out)
{
#pragma unroll
  for (int k = 0; k < N; k++) {
    const unsigned long long s = wave_sum(v[k]);
    if ((threadIdx.x & 63u) == 0) sh[(threadIdx.x >> 6) * N + k] = s;
  }
  __syncthreads();
  if (threadIdx.x < N) out[threadIdx.x] = sh[threadIdx.x] + sh[N + threadIdx.x] + sh[2 * N + threadIdx.x] + sh[3 * N + threadIdx.x];
}

// Counters stay in registers, the two histograms in 16 LDS copies (lane % 16),
// and a workgroup writes one record that k_feat_sum adds up.  With one copy,
// one LDS atomic per lane and counter and global atomics at the end, lanes and
// workgroups queued on the same addresses (300,007 rows of 4 to 64 entries:
// 133 us for this kernel and 106 for the entries'; 49 and 92 with only the
// global atomics left).
constexpr int FEAT_COPIES = 16;

__global__ __launch_bounds__(256) void k_feat_rows(uint32_t rows, const uint32_t *__restrict__ rp,
                                                   const uint32_t *__restrict__ ci,
                                                   feat_row_counters *__restrict__ out)
{
  __shared__ unsigned s_max[4];
  __shared__ uint32_t s_len[24][FEAT_COPIES + 1], s_nnz[16][FEAT_COPIES + 1]; // below 2^32: nnz and rows are
  __shared__ unsigned long long sh[4 * 7];
  const int t = threadIdx.x, copy = t % FEAT_COPIES;
  for (int i = t; i < 24 * (FEAT_COPIES + 1); i += 256) (&s_len[0][0])[i] = 0;
  for (int i = t; i < 16 * (FEAT_COPIES + 1); i += 256) (&s_nnz[0][0])[i] = 0;
  __syncthreads();
  unsigned long long sumsq = 0, empty = 0, big = 0, small = 0, gt64 = 0, span = 0, nonempty = 0;
  unsigned mx = 0;
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  for (uint64_t r = (uint64_t)blockIdx.x * 256u + t; r < rows; r += stride) {
    const uint32_t b = rp[r], len = rp[r + 1] - b;
    sumsq += (unsigned long long)len * len;
    mx = max(mx, len);
    if (len == 0) {
      empty++;
      atomicAdd(&s_len[0][copy], 1u);
      continue;
    }
    const uint32_t c0 = ci[b], c1 = ci[b + len - 1];
    const int lb = ilog2(len);
    atomicAdd(&s_len[min(23, lb + 1)][copy], 1u);
    atomicAdd(&s_nnz[min(15, lb)][copy], len);
    if (len > 4096) big += len;
    if (len <= 4) small += len;
    if (len > 64) gt64++;
    span += (unsigned long long)(c1 >= c0 ? c1 - c0 : c0 - c1) + 1;
    nonempty++;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, d, 64));
  if ((t & 63) == 0) s_max[t >> 6] = mx;
  feat_row_counters *o = out + blockIdx.x;
  const unsigned long long v[7] = {sumsq, empty, big, small, gt64, span, nonempty};
  block_sums(v, sh, &o->sumsq); // its barrier lies after the histograms' last atomics
  if (t == 0) o->max_len = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
  if (t < 24 + 16) {
    const uint32_t *h = t < 24 ? s_len[t] : s_nnz[t - 24];
    unsigned long long s = 0;
    for (int c = 0; c < FEAT_COPIES; c++) s += h[c];
    (t < 24 ? o->len_hist[t] : o->nnz_hist[t - 24]) = s;
  }
}

struct feat_thresholds {
  double t[7]; // 1e-4 4^k
};

// Bin of the relative distance num / denom among the thresholds.
__device__ __forceinline__ uint32_t distance_bin(double num, double denom, const feat_thresholds &th)
{
  const double d = num / denom;
  uint32_t k = 0;
#pragma unroll
  for (int q = 0; q < 7; q++) k += d >= th.t[q] ? 1u : 0u;
  return k;
}

// Tiles of ROWS_TILE entries, their rows found together (entry_rows.h).  Per
// entry the kernel is bound by its arithmetic: 64-bit products and compares
// and a division took 540 cycles per wave of entries.  EXACT53 (rows cols <=
// 2^53): the distance |c rows - r cols| is exact in double, so one fma gives
// it, and the quotient by rows cols comes from products with rounded
// reciprocals wherever these decide it: the bin is the exponent of d / 1e-4
// (the thresholds are powers of 4 there) unless the mantissa lies within
// 2^-20 of a power of two, the floor of 2^24 d is the product's unless an
// integer lies within 2^-26 (both products are within 2^-50 of the
// quotient).  The remaining entries divide.
template <bool EXACT53>
__global__ __launch_bounds__(ROWS_T) void k_feat_entries(uint32_t rows, uint32_t cols, uint64_t nnz, uint32_t ntiles,
                                                         const uint32_t *__restrict__ rp,
                                                         const uint32_t *__restrict__ ci, feat_thresholds th,
                                                         feat_entry_counters *__restrict__ out)
{
  __shared__ uint32_t mark[ROWS_TILE];
  __shared__ uint32_t shr[8];
  __shared__ unsigned long long sh[4 * 10];
  const uint32_t t = threadIdx.x;
  const double rowsd = (double)rows, colsd = (double)cols, denom = rowsd * colsd;
  const double inv24 = 16777216.0 / denom, inv4 = 1e4 / denom;
  uint32_t hist[8] = {0, 0, 0, 0, 0, 0, 0, 0}, diag = 0; // a lane sees fewer than 2^32 entries
  unsigned long long dsum = 0;
  // a run of consecutive tiles: only the first one's row is searched
  const uint32_t tile0 = (uint32_t)((uint64_t)ntiles * blockIdx.x / gridDim.x);
  const uint32_t tile1 = (uint32_t)((uint64_t)ntiles * (blockIdx.x + 1) / gridDim.x);
  uint32_t cn[ROWS_I];
  auto load = [&](uint32_t tile) {
    const uint64_t at = (uint64_t)tile * ROWS_TILE;
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++) cn[k] = ldg_stream(ci + min(at + k * ROWS_T + t, nnz - 1));
  };
  if (tile0 < tile1) load(tile0);
  uint32_t first = tile0 < tile1 ? block_row_of(rp, rows, tile0 * ROWS_TILE, shr + 4) : 0u;
  for (uint32_t tile = tile0; tile < tile1; tile++) {
    const uint32_t t0 = tile * ROWS_TILE;
    const uint64_t t1 = min(nnz, (uint64_t)t0 + ROWS_TILE);
    const uint32_t m = (uint32_t)(t1 - t0);
    uint32_t c[ROWS_I], row[ROWS_I];
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++) c[k] = cn[k];
    if (tile + 1 < tile1) load(tile + 1); // in flight during this tile
    tile_rows(rp, rows, first, t0, t1, mark, shr, row);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++) mark[t * ROWS_I + k] = row[k];
    __syncthreads();
    uint32_t lo = 0, hi = 0; // bins 0..3 and 4..7, a byte each (8 entries at most)
    uint32_t d24 = 0;        // 8 2^24 at most
#pragma unroll
    for (uint32_t k = 0; k < ROWS_I; k++) {
      const uint32_t l = k * ROWS_T + t;
      if (l >= m) break;
      const uint32_t r = mark[l];
      uint32_t bin;
      if constexpr (EXACT53) {
        const double num = fabs(__builtin_fma((double)c[k], rowsd, -((double)r * colsd)));
        const double v = num * inv4, q24 = num * inv24, fl = floor(q24), fr = q24 - fl;
        const int h = __double2hiint(v), e = (h >> 20) - 1023;
        const uint32_t mant = (uint32_t)h & 0xFFFFFu;
        bin = e < 0 ? 0u : min(7u, (uint32_t)(e >> 1) + 1u);
        if (e >= -1 && (mant == 0u || mant == 0xFFFFFu)) bin = distance_bin(num, denom, th);
        d24 += (uint32_t)(fr > 0x1p-26 && fr < 1.0 - 0x1p-26 ? fl : floor(num / denom * 16777216.0));
      } else {
        const uint64_t a = (uint64_t)c[k] * rows, b = (uint64_t)r * cols;
        const double num = (double)(a > b ? a - b : b - a);
        bin = distance_bin(num, denom, th);
        d24 += (uint32_t)(num / denom * 16777216.0);
      }
      const uint32_t one = 1u << (8u * (bin & 3u));
      lo += bin < 4u ? one : 0u;
      hi += bin < 4u ? 0u : one;
      diag += c[k] == r ? 1u : 0u;
    }
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
      hist[q] += (lo >> (8u * q)) & 255u;
      hist[4 + q] += (hi >> (8u * q)) & 255u;
    }
    dsum += d24;
    first = mark[m - 1u];
    __syncthreads(); // mark is reused
  }
  const unsigned long long v[10] = {hist[0], hist[1], hist[2], hist[3], hist[4], hist[5], hist[6], hist[7], dsum, diag};
  block_sums(v, sh, out[blockIdx.x].dist_hist);
}

// One workgroup per counter: the records' sum (the longest row: their maximum)
__global__ __launch_bounds__(256) void k_feat_sum(const unsigned long long *__restrict__ rrec, uint32_t nr,
                                                  const unsigned long long *__restrict__ erec, uint32_t ne,
                                                  unsigned long long *__restrict__ out)
{
  __shared__ unsigned long long sh[4];
  const uint32_t f = blockIdx.x, t = threadIdx.x;
  unsigned long long s = 0;
  if (f == FEAT_R - 1) {
    for (uint32_t i = t; i < nr; i += 256) s = max(s, rrec[(uint64_t)i * FEAT_R + f]);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s = max(s, (unsigned long long)__shfl_xor((long long)s, d, 64));
    if ((t & 63u) == 0) sh[t >> 6] = s;
    __syncthreads();
    s = max(max(sh[0], sh[1]), max(sh[2], sh[3]));
  } else {
    if (f < FEAT_R)
      for (uint32_t i = t; i < nr; i += 256) s += rrec[(uint64_t)i * FEAT_R + f];
    else
      for (uint32_t i = t; i < ne; i += 256) s += erec[(uint64_t)i * FEAT_E + (f - FEAT_R)];
    s = wave_sum(s);
    if ((t & 63u) == 0) sh[t >> 6] = s;
    __syncthreads();
    s = sh[0] + sh[1] + sh[2] + sh[3];
  }
  if (t == 0) out[f] = s;
}

} // namespace mfp

using namespace mfp;

extern "C" int mfp_matrix_features(mfp_matrix m, float *out)
{
  MFP_ARG(m && out, "null pointer");
  MFP_ARG(m->rows > 0 && m->cols > 0, "empty matrix");
  const uint32_t cus = (uint32_t)std::max(1, props().cu_count);
  const uint32_t gr = std::min<uint32_t>(2 * cus, ceil_div_u32(m->rows, 256));
  const uint32_t tiles = ceil_div_u32(m->nnz, ROWS_TILE), ge = std::min<uint32_t>(4 * cus, tiles);
  // the totals, the rows' records, the entries' records
  unsigned long long *dc = nullptr;
  MFP_CHECK(dmalloc((void **)&dc, (FEAT_R + FEAT_E + (uint64_t)gr * FEAT_R + (uint64_t)ge * FEAT_E) * 8));
  unsigned long long *rrec = dc + FEAT_R + FEAT_E, *erec = rrec + (uint64_t)gr * FEAT_R;
  struct {
    feat_row_counters r;
    feat_entry_counters e;
  } tot{};
  static_assert(sizeof(tot) == (FEAT_R + FEAT_E) * 8, "counters are u64 only");
  k_feat_rows<<<gr, 256>>>(m->rows, m->row_ptr, m->columns, (feat_row_counters *)rrec);
  if (ge) {
    feat_thresholds th;
    for (int k = 0; k < 7; k++) th.t[k] = 1e-4 * std::pow(4.0, k);
    const bool exact53 = (uint64_t)m->rows * m->cols <= 1ull << 53;
    (exact53 ? k_feat_entries<true> : k_feat_entries<false>)<<<ge, ROWS_T>>>(
        m->rows, m->cols, m->nnz, tiles, m->row_ptr, m->columns, th, (feat_entry_counters *)erec);
  }
  k_feat_sum<<<FEAT_R + FEAT_E, 256>>>(rrec, gr, erec, ge, dc);
  int st = MFP_OK;
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string("feature kernels: ") + hipGetErrorString(e));
    st = MFP_ERR_HIP;
  }
  if (st == MFP_OK) st = mfp_memcpy_d2h(&tot, dc, sizeof tot);
  {
    const free_scope scope(st == MFP_OK);
    dfree(dc);
  }
  MFP_CHECK(st);
  const feat_row_counters &h = tot.r;
  const feat_entry_counters &he = tot.e;

  const double rows = m->rows, cols = m->cols, nnz = (double)m->nnz;
  const double mean = nnz / rows;
  const double var = std::max(0.0, (double)h.sumsq / rows - mean * mean);
  const double sd = std::sqrt(var);
  const double cv = mean > 0 ? sd / mean : 0.0;
  const double nz = nnz > 0 ? nnz : 1.0;
  double f[64] = {0};
  f[0] = std::log2(rows + 1) / 32;
  f[1] = std::log2(cols + 1) / 32;
  f[2] = std::log2(nnz + 1) / 40;
  f[3] = std::log2(1 + mean) / 16;
  f[4] = std::log2(1 + (double)h.max_len) / 16;
  f[5] = std::min(cv, 32.0) / 32;
  f[6] = (double)h.empty / rows;
  f[7] = std::log2(1 + sd) / 16;
  for (int b = 0; b < 24; b++) f[8 + b] = (double)h.len_hist[b] / rows;
  for (int b = 0; b < 16; b++) f[32 + b] = (double)h.nnz_hist[b] / nz;
  for (int b = 0; b < 8; b++) f[48 + b] = (double)he.dist_hist[b] / nz;
  f[56] = (double)he.dist_sum / 16777216.0 / nz;
  f[57] = (double)he.diag / nz;
  f[58] = h.nonempty ? (double)h.span_sum / (double)h.nonempty / cols : 0.0;
  f[59] = nnz > 0 ? std::log2(rows * (double)h.max_len / nnz) / 16 : 0.0;
  f[60] = (double)h.nnz_big / nz;
  f[61] = (double)h.nnz_small / nz;
  f[62] = (double)h.rows_gt64 / rows;
  f[63] = 1.0;
  for (int i = 0; i < 64; i++) out[i] = (float)f[i];
  return MFP_OK;
}
