// SpMV kernels for gfx950: CSR-scalar, CSR-vector, CSR-Adaptive, ELL, COO,
// SCOO and the two hybrid ELL+COO forms.
//
// SpMV is bound by HBM bandwidth, so every kernel keeps several independent
// loads in flight per lane (loads are issued for a group of elements before
// any of them is used) and streams the matrix with nontemporal loads, which
// leaves L2 / Infinity Cache to the gathered x entries.
//
// Summation orders (bit-exact against the oracle's emulators where the
// kernel is deterministic):
//   CSR-scalar  sequential fma per row            (cpu_matrix_multiplier.cpp:20-61)
//   CSR-vector  G-lane strided fma + halving tree (cpu_matrix_multiplier.cpp:170-227, G=32)
//   ELL         sequential fma over the padded width
//   CSR-Adaptive: see k_csr_adaptive.
//   COO without rows above 64 entries: see coo_span (owner form).
// COO with longer rows, SCOO and the hybrids accumulate with atomics (order
// not fixed).
#include "kernels.h"
#include "mfp_internal.h"
#include "row_chunks.h"
#include "values16.h"
#include "wave64.h"

#include <hip/hip_ext.h>

#include <type_traits>

namespace mfp {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 16-byte value vectors and the matching column-index vectors.
template <typename T> struct vec16;
template <> struct vec16<float> {
  using V = f32x4;
  using I = u32x4;
  static constexpr uint32_t N = 4;
};
template <> struct vec16<double> {
  using V = f64x2;
  using I = u32x2;
  static constexpr uint32_t N = 2;
};

// ---------------------------------------------------------------------------
// CSR-scalar: one lane per row, as gpu_matrix_multiplier.cu:22-43, but the
// wave stages its rows' contiguous nnz range through LDS with coalesced loads
// so each lane then walks only its own row.  Order: sequential fma.
// The staging of a chunk is split in two so that no load waits behind
// another: the values and column indices of chunk k + 1 are issued before
// chunk k is summed, and their x gathers right after; every load sits at a
// clamped in-range offset, so none is predicated.  A lane reads its row
// from LDS eight elements at a time, so a long row pays the LDS latency once
// per eight fma.
// ---------------------------------------------------------------------------
constexpr uint32_t SCALAR_PER_LANE = 8, SCALAR_CHUNK = 64 * SCALAR_PER_LANE;

template <typename T>
__device__ __forceinline__ void scalar_stage_loads(const uint32_t *__restrict__ ci, const T *__restrict__ a,
                                                   uint32_t c0, uint32_t n, uint32_t lane, T (&av)[SCALAR_PER_LANE],
                                                   uint32_t (&cv)[SCALAR_PER_LANE])
{
#pragma unroll
  for (uint32_t k = 0; k < SCALAR_PER_LANE; k++) {
    const uint32_t j = min(lane + 64u * k, n - 1u); // n >= 1: a duplicate of the last element past the end
    av[k] = ldg_stream(a + c0 + j);
    cv[k] = ldg_stream(ci + c0 + j);
  }
}

template <typename T>
__global__ __launch_bounds__(64) void k_csr_scalar(uint32_t rows, const uint32_t *__restrict__ rp,
                                                   const uint32_t *__restrict__ ci,
                                                   const T *__restrict__ a, const T *__restrict__ x,
                                                   T *__restrict__ y)
{
  __shared__ T va[2][SCALAR_CHUNK];
  __shared__ T vx[2][SCALAR_CHUNK];
  const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t r0 = blk * 64u;
  const uint32_t lane = threadIdx.x;
  const uint32_t r = r0 + lane;
  const uint32_t rend = min(r0 + 64u, rows);
  const uint32_t rs = rp[min(r, rows)];
  const uint32_t re = rp[min(r + 1u, rows)];
  const uint32_t b = rp[r0], e = rp[rend];
  T dot = 0;
  if (b < e) {
    T av[SCALAR_PER_LANE], xv[SCALAR_PER_LANE];
    uint32_t cv[SCALAR_PER_LANE];
    scalar_stage_loads(ci, a, b, min(SCALAR_CHUNK, e - b), lane, av, cv);
#pragma unroll
    for (uint32_t k = 0; k < SCALAR_PER_LANE; k++) xv[k] = x[cv[k]];
    uint32_t buf = 0;
    for (uint32_t c0 = b; c0 < e; c0 += SCALAR_CHUNK, buf ^= 1u) {
      const uint32_t n = min(SCALAR_CHUNK, e - c0);
      // slots past n hold duplicates and are never read
#pragma unroll
      for (uint32_t k = 0; k < SCALAR_PER_LANE; k++) {
        va[buf][lane + 64u * k] = av[k];
        vx[buf][lane + 64u * k] = xv[k];
      }
      __syncthreads();
      const uint32_t c1 = c0 + SCALAR_CHUNK;
      const bool next = c1 < e; // uniform over the wave
      if (next) scalar_stage_loads(ci, a, c1, min(SCALAR_CHUNK, e - c1), lane, av, cv);
      const uint32_t lo = max(rs, c0), hi = min(re, c0 + n);
      const T *pa = va[buf] - c0, *px = vx[buf] - c0;
      uint32_t i = lo;
      for (; i + 8u <= hi; i += 8u) {
        T qa[8], qx[8];
#pragma unroll
        for (uint32_t q = 0; q < 8; q++) {
          qa[q] = pa[i + q];
          qx[q] = px[i + q];
        }
#pragma unroll
        for (uint32_t q = 0; q < 8; q++) dot = fma_t(qa[q], qx[q], dot);
      }
      for (; i < hi; i++) dot = fma_t(pa[i], px[i], dot);
      if (next) {
#pragma unroll
        for (uint32_t k = 0; k < SCALAR_PER_LANE; k++) xv[k] = x[cv[k]];
      }
      // the buffer written next is the one summed two chunks ago: the
      // barrier above already ordered those reads
    }
  }
  if (r < rows) y[r] = dot;
}

// ---------------------------------------------------------------------------
// CSR-vector: G lanes per row (G = 2..64; the reference uses a 32-lane warp,
// gpu_matrix_multiplier.cu:331-362).  Lane l accumulates elements l, l+G, ...
// with fma (four elements' loads issued together), then group_reduce<G>.
// ---------------------------------------------------------------------------
// Rows with at least eight elements per lane run a software pipeline: the
// values and column indices of the next eight are loaded (at clamped in-row
// offsets, so no load is predicated) before the x entries of the current
// eight are gathered and summed, so a long row waits for one memory latency
// per eight elements instead of two per four.
// The loops stand in the kernel itself: as a function that is inlined they
// take 65 VGPRs in FP32 instead of 48 and cost a wave per SIMD (800k entries in
// rows of 6, 34, 100: 7.3, 7.3, 5.6 us instead of 6.7, 6.8, 4.6).
template <typename T, int G>
__global__ __launch_bounds__(256) void k_csr_vector(uint32_t rows, const uint32_t *__restrict__ rp,
                                                    const uint32_t *__restrict__ ci,
                                                    const T *__restrict__ a, const T *__restrict__ x,
                                                    T *__restrict__ y)
{
  constexpr uint32_t U = 8;
  const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t row = (blk * 256u + threadIdx.x) / G;
  const uint32_t lane = threadIdx.x % G;
  T dot = 0;
  if (row < rows) {
    const uint32_t b = rp[row], e = rp[row + 1];
    uint32_t i = b + lane;
    if (i + (U - 1) * G < e) {
      T an[U];
      uint32_t cn[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) {
        an[u] = ldg_stream(a + i + u * G);
        cn[u] = ldg_stream(ci + i + u * G);
      }
      for (;;) {
        T ac[U];
        uint32_t cc[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
          ac[u] = an[u];
          cc[u] = cn[u];
        }
        const uint32_t inext = i + U * G;
        const bool more = inext + (U - 1) * G < e;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
          const uint32_t j = min(inext + u * G, e - 1u); // e > i: in range
          an[u] = ldg_stream(a + j);
          cn[u] = ldg_stream(ci + j);
        }
        T xv[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) xv[u] = x[cc[u]];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) dot = fma_t(ac[u], xv[u], dot);
        i = inext;
        if (!more) break;
      }
    }
    for (; i + 3u * G < e; i += 4u * G) {
      const T a0 = ldg_stream(a + i), a1 = ldg_stream(a + i + G);
      const T a2 = ldg_stream(a + i + 2 * G), a3 = ldg_stream(a + i + 3 * G);
      const uint32_t c0 = ldg_stream(ci + i), c1 = ldg_stream(ci + i + G);
      const uint32_t c2 = ldg_stream(ci + i + 2 * G), c3 = ldg_stream(ci + i + 3 * G);
      const T x0 = x[c0], x1 = x[c1], x2 = x[c2], x3 = x[c3];
      dot = fma_t(a0, x0, dot);
      dot = fma_t(a1, x1, dot);
      dot = fma_t(a2, x2, dot);
      dot = fma_t(a3, x3, dot);
    }
    for (; i < e; i += G) dot = fma_t(ldg_stream(a + i), x[ldg_stream(ci + i)], dot);
  }
  dot = group_reduce<G>(dot);
  if (lane == 0 && row < rows) y[row] = dot;
}

// The same sums from LDS.  A workgroup takes RB consecutive rows and stages
// as many whole ones as fit (a values and gathered x entries, CVL_K 16-byte
// vectors per lane, every load in flight before the first wait), then each
// group of G lanes sums its rows from there.  A longer row goes through LDS
// in chunks, the first group carrying its lanes' sums from one to the next.
//
// What bounds the kernel above is waiting: a wave of G = 64 lanes issues one
// load of values, one of columns and one of x entries per row of 34 entries,
// each after the last, and a row's 136 bytes are read in 4-byte loads.  Here
// a workgroup's loads are independent of its row lengths: 16 bytes per lane,
// two vectors of values and of columns, then their 8 (FP64: 4) gathers.
// Eight workgroups share a CU (16 KB of LDS, 48 to 60 VGPRs).  Where the
// rows fit at once, their values and columns are on the way before the row
// starts are staged, and the gathers go out together behind that barrier:
// 300,007 rows of 4 to 64 random entries 58.7 -> 53.3 us (FP64 72.5 -> 61.5);
// without the barrier between a wave's loads and its gathers 57 to 61 (71 to
// 72).  FP32, lanes from the mean, row by row -> from LDS: 27-point stencil of
// 100^3 121.7 -> 54.2 us, 5-point stencil of 1400^2 56.8 -> 22.5, those random
// rows 75.4 -> 53.1 (the gathers alone take 48.5), power-law 1M rows 342 -> 169
// (its 50,000-entry row is one wait per 1,984 entries instead of one per 8 per
// lane).  Larger chunks were slower: three vectors per lane 59.5 and four 70.6
// us on the 27-point stencil, against 55.5.
constexpr uint32_t CVL_K = 2, CVL_U = 2;
// entries of a listed row in flight, and of a staged row read from LDS together
constexpr uint32_t CVL_REST = 8;
template <typename T>
constexpr uint32_t CVL_STEP = sizeof(T) == 4 ? 8 : 4;
template <typename T>
struct cvl {
  static constexpr uint32_t N = vec16<T>::N, K = CVL_K, CAP = 256 * K * N;
  // chunk of a long row: a multiple of 64 lanes that fits at any alignment
  static constexpr uint32_t CHUNK = CAP - 64;
};

// Elements [base, base + n) into LDS at (element - base / N N); n + base % N <=
// CAP.  between() runs after the loads are issued and before the gathers.
template <typename T, typename F>
__device__ __forceinline__ void cvl_stage(uint32_t base, uint32_t n, const uint32_t *__restrict__ ci,
                                          const T *__restrict__ a, const T *__restrict__ x, T *sa, T *sx, F between)
{
  using VT = vec16<T>;
  constexpr uint32_t N = VT::N, K = cvl<T>::K;
  const uint32_t v0 = base / N, nv = (uint32_t)(((uint64_t)base + n + N - 1) / N) - v0;
  const typename VT::V *av = reinterpret_cast<const typename VT::V *>(a) + v0;
  const typename VT::I *cv = reinterpret_cast<const typename VT::I *>(ci) + v0;
  typename VT::V va[K], vx[K];
  typename VT::I vc[K];
#pragma unroll
  for (uint32_t k = 0; k < K; k++) {
    const uint32_t v = min(threadIdx.x + k * 256u, nv - 1u);
    va[k] = ldg_stream(av + v);
    vc[k] = ldg_stream(cv + v);
  }
  between();
  const uint32_t lo = base - v0 * N, hi = lo + n; // the vectors' elements that count
#pragma unroll
  for (uint32_t k = 0; k < K; k++)
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
      const uint32_t e = min(threadIdx.x + k * 256u, nv - 1u) * N + j;
      vx[k][j] = x[e >= lo && e < hi ? vc[k][j] : 0u];
    }
#pragma unroll
  for (uint32_t k = 0; k < K; k++) {
    const uint32_t v = threadIdx.x + k * 256u;
    if (v < nv) {
      reinterpret_cast<typename VT::V *>(sa)[v] = va[k];
      reinterpret_cast<typename VT::V *>(sx)[v] = vx[k];
    }
  }
}

// One lane's sum of the row [b, e): its elements in k_csr_vector's order,
// CVL_REST at a time.
template <typename T, int G>
__device__ __forceinline__ T csr_vector_row(uint32_t b, uint32_t e, uint32_t lane, const uint32_t *__restrict__ ci,
                                            const T *__restrict__ a, const T *__restrict__ x)
{
  constexpr uint32_t U = CVL_REST;
  uint32_t left = e - b > lane ? (e - b - lane - 1u) / G + 1u : 0u; // counted down: positions may end at 2^32
  uint32_t i = b + lane;
  T dot = 0;
  if (left >= U) {
    uint32_t next[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) next[u] = ldg_stream(ci + i + u * G);
    for (; left >= U; left -= U, i += U * G) {
      // the gathers, this round's values and the next round's columns together
      T v[U], xv[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) xv[u] = x[next[u]];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) {
        v[u] = ldg_stream(a + i + u * G);
        next[u] = ldg_stream(ci + min(i + (U + u) * G, e - 1u)); // past the row: not used
      }
#pragma unroll
      for (uint32_t u = 0; u < U; u++) dot = fma_t(v[u], xv[u], dot);
    }
  }
  for (; left; left--, i += G) dot = fma_t(ldg_stream(a + i), x[ldg_stream(ci + i)], dot);
  return dot;
}

// The first `extra` workgroups (a multiple of 8) sum the nlist listed blocks of
// rows as k_csr_vector does, `lists` lanes each; mask has a bit for each block
// of the list (csr_vector_layout_build).
template <typename T, int G>
__global__ __launch_bounds__(256, 8) void k_csr_vector_lds(uint32_t rows, uint32_t RB, uint32_t extra, uint32_t lists,
                                                        uint32_t nlist, const uint32_t *__restrict__ list,
                                                        const uint32_t *__restrict__ mask,
                                                        const uint32_t *__restrict__ rp,
                                                        const uint32_t *__restrict__ ci,
                                                        const T *__restrict__ a, const T *__restrict__ x,
                                                        T *__restrict__ y)
{
  constexpr uint32_t N = cvl<T>::N, CAP = cvl<T>::CAP, CHUNK = cvl<T>::CHUNK;
  __shared__ __align__(16) T sa[CAP];
  __shared__ __align__(16) T sx[CAP];
  __shared__ uint32_t rs[257];
  const uint32_t tid = threadIdx.x;
  if (blockIdx.x < extra) {
    const uint32_t per = (RB * G + lists - 1u) / lists, h = blockIdx.x / per;
    if (h >= nlist || tid >= lists) return;
    const uint32_t l0 = list[h] * RB, lr = (blockIdx.x % per * lists + tid) / G, row = l0 + lr;
    const bool ok = lr < min(RB, rows - l0);
    T dot = ok ? csr_vector_row<T, G>(rp[row], rp[row + 1], tid % G, ci, a, x) : (T)0;
    dot = group_reduce<G>(dot);
    if (ok && tid % G == 0) y[row] = dot;
    return;
  }
  const uint32_t blk = xcd_block(blockIdx.x - extra, gridDim.x - extra), r0 = blk * RB; // RB <= 256
  const uint32_t nr = min(RB, rows - r0);
  const uint32_t p = tid <= nr ? rp[r0 + tid] : 0u, first = rp[r0], last = rp[r0 + nr];
  const bool all = last - first <= CAP - first % N; // the usual case: every row fits at once
  if (!all && nlist && ((mask[blk >> 5] >> (blk & 31u)) & 1u)) return; // listed
  auto row_starts = [&] {
    if (tid <= nr) rs[tid] = p;
    if (tid == 0 && nr == 256u) rs[256] = last;
    __syncthreads();
  };
  if (all && last > first) {
    cvl_stage(first, last - first, ci, a, x, sa, sx, row_starts);
    __syncthreads();
  } else {
    row_starts();
  }
  const uint32_t lane = tid % G, grp = tid / G;
  for (uint32_t cur = 0; cur < nr;) {
    const uint32_t base = rs[cur], off = base % N;
    if (!all && rs[cur + 1] - base > CAP - off) {
      const uint32_t e = rs[cur + 1];
      T dot = 0;
      for_row_chunks(base, e, CHUNK, [&](uint32_t c0, uint32_t n) {
        cvl_stage(c0, n, ci, a, x, sa, sx, [] {});
        __syncthreads();
        if (tid < G) {
          const uint32_t sh = c0 % N;
          uint32_t i = lane;
          for (; i + 7u * G < n; i += 8u * G) {
            T qa[8], qx[8];
#pragma unroll
            for (uint32_t q = 0; q < 8; q++) {
              qa[q] = sa[sh + i + q * G];
              qx[q] = sx[sh + i + q * G];
            }
#pragma unroll
            for (uint32_t q = 0; q < 8; q++) dot = fma_t(qa[q], qx[q], dot);
          }
          for (; i < n; i += G) dot = fma_t(sa[sh + i], sx[sh + i], dot);
        }
        __syncthreads();
      });
      if (tid < 64u) { // the first group's wave
        dot = group_reduce<G>(dot);
        if (tid == 0) y[r0 + cur] = dot;
      }
      cur++;
      continue;
    }
    // whole rows that fit behind base
    uint32_t end = nr;
    if (!all) {
      end = cur + (uint32_t)__syncthreads_count(tid >= cur && tid < nr && rs[tid + 1] - base <= CAP - off);
      const uint32_t n = rs[end] - base;
      if (n) cvl_stage(base, n, ci, a, x, sa, sx, [] {});
      __syncthreads();
    }
    const uint32_t org = base - off;
    // U rows of a group side by side; the wave's groups stay together
    constexpr uint32_t ST = 256u / G, U = CVL_U;
    for (uint32_t r = cur + grp; r - grp < end; r += U * ST) {
      uint32_t b[U], e[U];
      T dot[U], qa[U], qx[U];
#pragma unroll
      for (uint32_t q = 0; q < U; q++) {
        const uint32_t rr = min(r + q * ST, end - 1u);
        b[q] = rs[rr] - org + lane;
        e[q] = rs[rr + 1] - org;
      }
#pragma unroll
      for (uint32_t q = 0; q < U; q++) {
        const uint32_t i = min(b[q], CAP - 1u);
        qa[q] = sa[i];
        qx[q] = sx[i];
      }
#pragma unroll
      for (uint32_t q = 0; q < U; q++) dot[q] = b[q] < e[q] ? fma_t(qa[q], qx[q], (T)0) : (T)0;
#pragma unroll
      for (uint32_t q = 0; q < U; q++) {
        constexpr uint32_t S = CVL_STEP<T>;
        uint32_t i = b[q] + G;
        for (; i + (S - 1u) * G < e[q]; i += S * G) { // not one LDS latency per element
          T ra[S], rx[S];
#pragma unroll
          for (uint32_t k = 0; k < S; k++) {
            ra[k] = sa[i + k * G];
            rx[k] = sx[i + k * G];
          }
#pragma unroll
          for (uint32_t k = 0; k < S; k++) dot[q] = fma_t(ra[k], rx[k], dot[q]);
        }
        for (; i < e[q]; i += G) dot[q] = fma_t(sa[i], sx[i], dot[q]);
      }
#pragma unroll
      for (uint32_t q = 0; q < U; q++) dot[q] = group_reduce<G>(dot[q]);
#pragma unroll
      for (uint32_t q = 0; q < U; q++)
        if (lane == 0 && r + q * ST < end) y[r0 + r + q * ST] = dot[q];
    }
    if (all) return;
    __syncthreads();
    cur = end;
  }
}

// ---------------------------------------------------------------------------
// CSR-Adaptive (csr_adaptive_spmv.cu:26-178 redesigned for 256-lane
// workgroups and LDS-sized row blocks).
//   multi-row block  (CSR-Stream): the block's nnz range is read with 16-byte
//     vector loads (K vectors per lane, all in flight together), rounded
//     products a*x staged in LDS (up to nnz_per_wg of them).  The reduction
//     is balanced whatever the row lengths: lane i sums the products
//     [i*E, i*E + E) (E = ceil(nnz_per_wg / 256)) left to right, restarting
//     at every row boundary; rows inside one lane finish there, and the
//     partial a lane carries into the next enters a 256-lane Hillis-Steele
//     segmented scan; a row ending in lane j that began earlier is
//     scan[j-1] + lane j's partial.
//     A block spends its time waiting, phase after phase, so the phases are
//     kept short and side by side: the row starts are loaded beside the
//     entries (they came after the products), the gathers go out together
//     behind the barrier that stages them and are in flight while the rows
//     are searched, products lie where the lanes' runs read them from
//     different banks, and the scan takes as many steps as the longest
//     carried row needs, one barrier each (it took eight of two).  27-point
//     grid of 100^3 f32 58.6 -> 52.5 us, f64 93.4 -> 67.9; 300k rows of 34
//     random entries f32 60.4 -> 51.2, f64 71.4 -> 54.6; 1M power-law rows f32
//     84.4 -> 79.0, f64 139 -> 138 (x of 8 MB is past an XCD's L2: its gathers
//     alone take 125).  Gathers before the barrier: 52.6, 72.0, 52.8, 57.4,
//     81.6 and 139 us.
//   single-row block (CSR-Vector/VectorL): 256 lanes strided with fma, a
//     64-lane halving tree per wave, then a halving tree over the 4 waves.
//   rows longer than long_row: split into `chunk`-element pieces, one
//     workgroup each, reduced like a single-row block; k_adaptive_finish
//     (launched next on the same stream) adds a row's pieces left to right.
//     The pieces are dispatched first, round-robin over the XCDs.
// ---------------------------------------------------------------------------
constexpr uint32_t AD_T = 256;

template <typename T>
__device__ __forceinline__ T wg_row_sum(const uint32_t *__restrict__ ci, const T *__restrict__ a,
                                        const T *__restrict__ x, uint32_t b, uint32_t e, T *wsum)
{
  T d = 0;
  uint32_t i = b + threadIdx.x;
  for (; i + 3 * AD_T < e; i += 4 * AD_T) {
    const T a0 = ldg_stream(a + i), a1 = ldg_stream(a + i + AD_T);
    const T a2 = ldg_stream(a + i + 2 * AD_T), a3 = ldg_stream(a + i + 3 * AD_T);
    const uint32_t c0 = ldg_stream(ci + i), c1 = ldg_stream(ci + i + AD_T);
    const uint32_t c2 = ldg_stream(ci + i + 2 * AD_T), c3 = ldg_stream(ci + i + 3 * AD_T);
    const T x0 = x[c0], x1 = x[c1], x2 = x[c2], x3 = x[c3];
    d = fma_t(a0, x0, d);
    d = fma_t(a1, x1, d);
    d = fma_t(a2, x2, d);
    d = fma_t(a3, x3, d);
  }
  for (; i < e; i += AD_T) d = fma_t(ldg_stream(a + i), x[ldg_stream(ci + i)], d);
  d = group_reduce<64>(d);
  if ((threadIdx.x & 63u) == 0) wsum[threadIdx.x >> 6] = d;
  __syncthreads();
  T r = 0;
  if (threadIdx.x == 0) {
    const T w0 = wsum[0] + wsum[2];
    const T w1 = wsum[1] + wsum[3];
    r = w0 + w1;
  }
  return r;
}

// Place of staged product e: lanes read runs of 8 (FP32) or 4 (FP64) side by
// side, and a gap after each keeps their reads on different banks.  gap is the
// log2 of the run; ADAPTIVE_NO_GAP leaves the gaps out.
constexpr uint32_t ADAPTIVE_NO_GAP = 31;
__host__ __device__ constexpr uint32_t adaptive_slot(uint32_t e, uint32_t gap) { return e + (e >> gap); }

// bytes of the staged products, a multiple of 16
template <typename T>
__host__ __device__ constexpr uint32_t adaptive_products(uint32_t W, uint32_t gap)
{
  return (adaptive_slot(W, gap) * (uint32_t)sizeof(T) + 15u) & ~15u;
}

// A workgroup takes one item: the pieces of long rows first, then the row
// blocks in XCD order.  A batch's blocks differ in cost from one member to the
// next, so there the XCDs take runs of 64, as workgroups end: 512 matrices,
// f32, 1,468 us with a range per XCD, 1,341 in runs; 64 257 and 212.  (A fixed
// grid that walks the items in runs drifts apart and loses x in the L2s: 2,477
// us for the 512, 228 for the 64.)  One matrix keeps a range per XCD (300k rows
// within a band of 1%: 28.3 us, 29.3 in runs of 64 and 32 in runs of 16).
template <typename T, uint32_t K, bool BATCH>
__global__ __launch_bounds__(AD_T) void k_csr_adaptive(
    const uint32_t *__restrict__ rp, const uint32_t *__restrict__ ci, const T *__restrict__ a,
    const T *__restrict__ x, T *__restrict__ y, const uint32_t *__restrict__ blocks,
    uint32_t nnz_per_wg, uint32_t long_row, const uint4 *__restrict__ chunks, uint32_t nchunks,
    uint32_t nchunks_pad, uint32_t chunk, uint32_t gap, T *__restrict__ partials)
{
  using VT = vec16<T>;
  constexpr uint32_t N = VT::N;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *cache = reinterpret_cast<T *>(smem_raw); // staged products (nnz_per_wg, by adaptive_slot)
  // block-relative row starts (nnz_per_wg + 2)
  uint32_t *rs = reinterpret_cast<uint32_t *>(smem_raw + adaptive_products<T>(nnz_per_wg, gap));
  __shared__ T wsum[4];
  __shared__ T sv[2 * AD_T];
  __shared__ uint32_t wsteps[4];
  const uint32_t hw = blockIdx.x;
  const uint32_t tid = threadIdx.x;

  if (hw < nchunks_pad) {
    if (hw >= nchunks) return;
    const uint4 c4 = chunks[hw]; // {row, piece, first item, pieces}
    const uint32_t s = rp[c4.x], e = rp[c4.x + 1];
    const uint32_t cb = s + c4.y * chunk;
    const uint32_t ce = min(e, cb + chunk);
    const T p = wg_row_sum(ci, a, x, cb, ce, wsum);
    if (tid == 0) partials[c4.z + c4.y] = p;
    return;
  }

  const uint32_t b = hw - nchunks_pad, nb = gridDim.x - nchunks_pad;
  const uint32_t item = BATCH ? xcd_runs(b, nb, BATCH_RUN) : xcd_block(b, nb);
  const uint32_t r0 = blocks[item], r1 = blocks[item + 1];
  if (r1 <= r0) return;
  if (r1 - r0 == 1) {
    const uint32_t s = rp[r0], e = rp[r0 + 1];
    if (e - s > long_row) return; // handled by the chunk items
    const T d = wg_row_sum(ci, a, x, s, e, wsum);
    if (tid == 0) y[r0] = d;
    return;
  }

  // CSR-Stream: vectors [v0, v1) cover the block's elements [base, base + n)
  const uint32_t base = rp[r0];
  const uint32_t n = rp[r1] - base;
  const uint32_t v0 = base / N, v1 = (base + n + N - 1) / N;
  const typename VT::V *av = reinterpret_cast<const typename VT::V *>(a);
  const typename VT::I *cv = reinterpret_cast<const typename VT::I *>(ci);
  typename VT::V va[K];
  typename VT::I vc[K];
#pragma unroll
  for (uint32_t k = 0; k < K; k++) {
    const uint32_t v = v0 + tid + k * AD_T;
    if (v < v1) {
      va[k] = ldg_stream(av + v);
      vc[k] = ldg_stream(cv + v);
    }
  }
  // EARLY: the products are finished before the row starts are staged.  With 16
  // vectors per lane, x entries held over the search take 178 VGPRs in FP64 and
  // leave a CU two workgroups of three (4,096 entries per workgroup, 27-point
  // 100^3: 118 us, 98 so); the smaller forms gain from it.
  constexpr bool EARLY = sizeof(T) == 8 && K >= 16;
  T xv[K][N];
  if constexpr (EARLY) {
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
      const uint32_t v = v0 + tid + k * AD_T;
#pragma unroll
      for (uint32_t j = 0; j < N; j++) {
        const uint32_t e = v * N + j;
        xv[k][j] = (v < v1 && e >= base && e < base + n) ? x[vc[k][j]] : (T)0;
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
      const uint32_t v = v0 + tid + k * AD_T;
#pragma unroll
      for (uint32_t j = 0; j < N; j++) {
        const uint32_t e = v * N + j;
        if (v < v1 && e >= base && e < base + n) cache[adaptive_slot(e - base, gap)] = va[k][j] * xv[k][j];
      }
    }
  }
  // the row starts are loaded beside the entries; the gathers go out together
  // behind their barrier and are in flight while the rows are searched
  const uint32_t nr = r1 - r0;
  const uint32_t p0 = tid <= nr ? rp[r0 + tid] : 0u, p1 = tid + AD_T <= nr ? rp[r0 + tid + AD_T] : 0u;
  // block-relative row starts rs[0..nr]
  if (tid <= nr) rs[tid] = p0 - base;
  if (tid + AD_T <= nr) rs[tid + AD_T] = p1 - base;
  for (uint32_t lr = tid + 2 * AD_T; lr <= nr; lr += AD_T) rs[lr] = rp[r0 + lr] - base;
  __syncthreads();
  if (!EARLY && n) { // without entries x may be empty
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
      const uint32_t v = v0 + tid + k * AD_T;
#pragma unroll
      for (uint32_t j = 0; j < N; j++) {
        const uint32_t e = v * N + j;
        xv[k][j] = x[v < v1 && e >= base && e < base + n ? vc[k][j] : 0u]; // outside the block: x[0], not used
      }
    }
  }
  for (uint32_t lr = tid; lr < nr; lr += AD_T)
    if (rs[lr] == rs[lr + 1]) y[r0 + lr] = (T)0; // empty rows

  // lane's run [e0, e1): sums split at row boundaries
  const uint32_t E = (nnz_per_wg + AD_T - 1) / AD_T;
  const uint32_t e0 = tid * E;
  const uint32_t e1 = min(n, e0 + E);
  uint32_t cur = 0;
  if (e0 < e1) {
    uint32_t hi = nr; // rs[cur] <= e0 < rs[hi]
    while (hi - cur > 1) {
      const uint32_t mid = (cur + hi) >> 1;
      if (rs[mid] <= e0)
        cur = mid;
      else
        hi = mid;
    }
  }
  if constexpr (!EARLY) {
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
      const uint32_t v = v0 + tid + k * AD_T;
#pragma unroll
      for (uint32_t j = 0; j < N; j++) {
        const uint32_t e = v * N + j;
        if (v < v1 && e >= base && e < base + n) cache[adaptive_slot(e - base, gap)] = va[k][j] * xv[k][j];
      }
    }
  }
  __syncthreads();
  T carry_v = 0;     // partial carried into the next lane
  uint32_t back = 0; // lanes back to the one where the carried row begins
  uint32_t frow = 0xFFFFFFFFu;
  T fval = 0;
  if (e0 < e1) {
    uint32_t cur_start = rs[cur], cur_end = rs[cur + 1];
    uint32_t seg = e0;
    T d = 0;
    for (uint32_t e = e0; e < e1; e++) {
      while (cur_end <= e) {
        if (seg < e) {
          if (seg == cur_start) {
            y[r0 + cur] = d;
          } else {
            frow = cur;
            fval = d;
          }
        }
        d = 0;
        seg = e;
        cur++;
        cur_start = cur_end;
        cur_end = rs[cur + 1];
      }
      d = d + cache[adaptive_slot(e, gap)];
    }
    const bool starts = seg == cur_start;
    if (e1 == cur_end) {
      if (starts) {
        y[r0 + cur] = d;
      } else {
        frow = cur;
        fval = d;
      }
    } else {
      carry_v = d;
      if (!starts) back = tid - cur_start / E;
    }
  }
  // segmented inclusive scan of the carried partials (Hillis-Steele), as many
  // steps as the longest way back takes; the two halves of sv take turns
  uint32_t steps = 0;
  while (__ballot(back >= (1u << steps))) steps++;
  sv[tid] = carry_v;
  if ((tid & 63u) == 0) wsteps[tid >> 6] = steps;
  __syncthreads();
  steps = max(max(wsteps[0], wsteps[1]), max(wsteps[2], wsteps[3]));
  for (uint32_t i = 0; i < steps; i++) {
    const uint32_t off = 1u << i, from = (i & 1u) * AD_T + tid;
    T v = sv[from];
    if (back >= off) v = sv[from - off] + v;
    sv[AD_T - (i & 1u) * AD_T + tid] = v;
    __syncthreads();
  }
  if (frow != 0xFFFFFFFFu) y[r0 + frow] = sv[(steps & 1u) * AD_T + tid - 1] + fval;
}

// One lane per long row: add its pieces left to right.
// p[0] + p[stride] + ... + p[(n - 1) stride], added left to right (n >= 1).
// Loads go out eight at a time with clamped indices, so none waits on the
// sum before it is issued; the additions keep the order.
template <typename T>
__device__ __forceinline__ T sum_in_order(const T *__restrict__ p, uint32_t n, uint64_t stride)
{
  T d = p[0];
  for (uint32_t k = 1; k < n; k += 8) {
    T q[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) q[j] = p[(uint64_t)min(k + j, n - 1) * stride];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) d = (k + j < n) ? d + q[j] : d;
  }
  return d;
}

template <typename T>
__global__ void k_adaptive_finish(const uint4 *__restrict__ chunks, uint32_t nchunks,
                                  const T *__restrict__ partials, T *__restrict__ y)
{
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nchunks) return;
  const uint4 c4 = chunks[j];
  if (c4.y != 0) return;
  y[c4.x] = sum_in_order(partials + c4.z, c4.w, 1);
}

// ---------------------------------------------------------------------------
// ELL: one lane per row, data[row + k*rows] (coalesced across lanes by
// construction), sequential fma over the padded width
// (gpu_matrix_multiplier.cu:450-471).  ATOMIC adds instead of storing (the
// fused hybrid).
// ---------------------------------------------------------------------------
template <typename T, bool ATOMIC>
__device__ __forceinline__ void ell_row(uint32_t r, uint32_t rows, uint32_t w,
                                        const uint32_t *__restrict__ ec, const T *__restrict__ ev,
                                        const T *__restrict__ x, T *__restrict__ y)
{
  T d = 0;
  uint64_t o = r;
  // groups of 8 slots, then 4 / 2 / 1: each group's loads are all in flight
  // before the first fma, and the fma order stays slot order
  auto group = [&](auto n_const) {
    constexpr uint32_t N = decltype(n_const)::value;
    T a[N];
    uint32_t c[N];
#pragma unroll
    for (uint32_t q = 0; q < N; q++) {
      a[q] = ldg_stream(ev + o + (uint64_t)q * rows);
      c[q] = ldg_stream(ec + o + (uint64_t)q * rows);
    }
    T xv[N];
#pragma unroll
    for (uint32_t q = 0; q < N; q++) xv[q] = x[c[q]];
#pragma unroll
    for (uint32_t q = 0; q < N; q++) d = fma_t(a[q], xv[q], d);
    o += (uint64_t)N * rows;
  };
  uint32_t k = 0;
  for (; k + 8 <= w; k += 8) group(std::integral_constant<uint32_t, 8>{});
  if (k + 4 <= w) {
    group(std::integral_constant<uint32_t, 4>{});
    k += 4;
  }
  if (k + 2 <= w) {
    group(std::integral_constant<uint32_t, 2>{});
    k += 2;
  }
  if (k < w) group(std::integral_constant<uint32_t, 1>{});
  if constexpr (ATOMIC)
    unsafeAtomicAdd(y + r, d);
  else
    y[r] = d;
}

template <typename T>
__global__ __launch_bounds__(256) void k_ell(uint32_t rows, uint32_t w, const uint32_t *__restrict__ ec,
                                             const T *__restrict__ ev, const T *__restrict__ x,
                                             T *__restrict__ y)
{
  const uint32_t r = xcd_block(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (r < rows) ell_row<T, false>(r, rows, w, ec, ev, x, y);
}

// FP32 / FP64 ELL over a 64-row sliced layout with 16-bit column offsets
// (plans created with MFP_TUNE_ELL_PACKED).  Slots 4j .. 4j + 3 of row r are
// value word j (four values) and offset word j (four u16); with
// u = (r / 64) w4 + j, the offset word is at u 64 + r % 64, and the value
// word is a float4 at u 64 + r % 64 (FP32) or two double2 halves, slots
// 4j, 4j + 1 at 2u 64 + r % 64 and 4j + 2, 4j + 3 at (2u + 1) 64 + r % 64
// (FP64), so every 16-byte load of a wave reads 1 KiB contiguous.  A slot's
// column is base[r / 64] + its offset.  A slot takes 6 bytes instead of 8
// (FP64: 10 instead of 12).  The fma order is k_ell's, slots 0 .. w - 1 (the
// slots past w that fill the last word are skipped); a padding slot adds
// 0 x x[base].
typedef uint16_t pk_u16x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T> struct pk_word;
template <> struct pk_word<float> {
  typedef f32x4 type;
  typedef f32x4 unit; // the array's element: one word
  static __device__ __forceinline__ type load(const unit *__restrict__ v, uint64_t u, uint32_t lr)
  {
    return __builtin_nontemporal_load(v + u * 64u + lr);
  }
};
template <> struct pk_word<double> {
  typedef f64x4 type;
  typedef f64x2 unit; // the array's element: half a word
  static __device__ __forceinline__ type load(const unit *__restrict__ v, uint64_t u, uint32_t lr)
  {
    const f64x2 lo = __builtin_nontemporal_load(v + u * 128u + lr);
    const f64x2 hi = __builtin_nontemporal_load(v + u * 128u + 64u + lr);
    return type{lo.x, lo.y, hi.x, hi.y};
  }
};

template <typename T>
__global__ __launch_bounds__(256) void k_ell_pk(uint32_t rows, uint32_t w, uint32_t w4,
                                                const uint32_t *__restrict__ base,
                                                const typename pk_word<T>::unit *__restrict__ val,
                                                const pk_u16x4 *__restrict__ off, const T *__restrict__ x,
                                                T *__restrict__ y)
{
  typedef typename pk_word<T>::type V;
  const uint32_t r = xcd_block(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (r >= rows) return;
  const uint32_t blk = r >> 6, lr = r & 63u;
  const T *__restrict__ xb = x + base[blk];
  T d = 0;
  // N words of 4 slots, every load of the group in flight before the first fma
  auto group = [&](uint32_t j, auto n_const) {
    constexpr uint32_t N = decltype(n_const)::value;
    pk_u16x4 o[N];
    V v[N];
#pragma unroll
    for (uint32_t q = 0; q < N; q++) {
      const uint64_t u = (uint64_t)blk * w4 + j + q;
      o[q] = __builtin_nontemporal_load(off + u * 64u + lr);
      v[q] = pk_word<T>::load(val, u, lr);
    }
    T xv[N][4];
#pragma unroll
    for (uint32_t q = 0; q < N; q++)
#pragma unroll
      for (uint32_t e = 0; e < 4; e++) xv[q][e] = xb[o[q][e]];
#pragma unroll
    for (uint32_t q = 0; q < N; q++)
#pragma unroll
      for (uint32_t e = 0; e < 4; e++)
        if (4u * (j + q) + e < w) d = fma_t(v[q][e], xv[q][e], d);
  };
  uint32_t j = 0;
  // a row of 5 to 8 words (up to 32 slots) is one group, every load of the
  // row in flight before the first gather (3D 27-point stencil, 7 words:
  // FP32 62.2 against 64.0 us in groups of 4, 2 and 1, FP64 111.5 against
  // 113.5 us, though FP64 then holds 148 VGPRs, 3 waves per SIMD)
  if (w4 >= 5 && w4 <= 8) {
    switch (w4) {
    case 8: group(0, std::integral_constant<uint32_t, 8>{}); break;
    case 7: group(0, std::integral_constant<uint32_t, 7>{}); break;
    case 6: group(0, std::integral_constant<uint32_t, 6>{}); break;
    default: group(0, std::integral_constant<uint32_t, 5>{}); break;
    }
    j = w4;
  }
  for (; j + 4 <= w4; j += 4) group(j, std::integral_constant<uint32_t, 4>{});
  if (j + 2 <= w4) {
    group(j, std::integral_constant<uint32_t, 2>{});
    j += 2;
  }
  if (j < w4) group(j, std::integral_constant<uint32_t, 1>{});
  y[r] = d;
}

// The packed layout of k_ell_pk from CSR: a thread per row (rows rounded up
// to 64; the extra rows and the slots past a row's length hold value 0,
// offset 0).
template <typename T>
__global__ void k_ell_pk_build(uint32_t rows, uint32_t stride, const uint32_t *__restrict__ rp,
                               const uint32_t *__restrict__ ci, const T *__restrict__ a, uint32_t w4,
                               const uint32_t *__restrict__ base, T *__restrict__ val,
                               uint16_t *__restrict__ off)
{
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= stride) return;
  const uint32_t s = r < rows ? rp[r] : 0u, len = r < rows ? rp[r + 1] - s : 0u;
  const uint32_t blk = r >> 6, lr = r & 63u, b0 = base[blk];
  for (uint32_t k = 0; k < 4u * w4; k++) {
    const bool in = k < len;
    const uint64_t u = (uint64_t)blk * w4 + k / 4u;
    off[(u * 64u + lr) * 4u + k % 4u] = in ? (uint16_t)(ci[s + k] - b0) : (uint16_t)0;
    // FP32: word u of row lr is one float4; FP64: two double2 halves
    const uint64_t at = sizeof(T) == 4 ? (u * 64u + lr) * 4u + k % 4u
                                       : ((u * 2u + (k % 4u) / 2u) * 64u + lr) * 2u + k % 2u;
    val[at] = in ? a[s + k] : (T)0;
  }
}

// y += t, element-wise (the host-COO hybrid's merge of the tail sums,
// gpu_matrix_multiplier.cu:1098-1108)
template <typename T>
__global__ __launch_bounds__(256) void k_vec_add(uint32_t n, const T *__restrict__ t, T *__restrict__ y)
{
  const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (i < n) y[i] = y[i] + t[i];
}

// ---------------------------------------------------------------------------
// COO (gpu_matrix_multiplier.cu:622-638): a wave takes COO_SPAN consecutive
// (row-sorted) entries, four per lane in 16-byte loads, all in flight
// together.  A lane adds up its runs of equal rows, one segmented scan over
// the lanes joins the runs that cross them, and every run leaves as one
// result.
//   atomic form  each run is added to y, which starts at zero
//   owner form   (no row above COO_AHEAD entries) the wave that holds a row's
//                first entry stores the row: it also reads the entries past
//                its span that the longest row can have there.  Nothing is
//                zeroed first and nothing is atomic, so an SpMV is one launch.
//                FP32, before -> now: 65,536 rows of 5 7.4 -> 3.6 us (two
//                launches of about 3.7), 5-point stencil 1400^2 34.3 -> 27.3,
//                27-point 100^3 75.1 -> 65.8, 300,007 rows of 4 to 64 75.0 ->
//                69.6; FP64 6.9 -> 3.6, 45.8 -> 38.4, 100.9 -> 98.8, 83.9 ->
//                80.7 (27-point 100^3 with 64 entries read ahead: 104.1).
//                With longer rows, walked on past the look-ahead, it lost:
//                rows of up to 500, 72.5 against 57.2 us.
// The atomic form was 64 entries per scan, four scans per wave: power-law 1M
// rows 99.2 -> 86.9 us.
// ---------------------------------------------------------------------------
constexpr uint32_t COO_SPAN = 256, COO_AHEAD = 64, COO_NONE = 0xFFFFFFFFu;

// ahead (owner form): entries that the longest row can have past its span
template <typename T, bool OWNER>
__device__ __forceinline__ void coo_span(uint64_t w0, uint64_t n, uint32_t ahead, const uint32_t *__restrict__ cr,
                                         const uint32_t *__restrict__ cc, const T *__restrict__ cv,
                                         const T *__restrict__ x, T *__restrict__ y)
{
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t i0 = w0 + 4u * lane, ia = w0 + COO_SPAN + lane;
  uint32_t r[4] = {COO_NONE, COO_NONE, COO_NONE, COO_NONE}, c[4] = {0, 0, 0, 0};
  T v[4] = {0, 0, 0, 0};
  // the entry before the span (lane 0), the entries after it
  uint32_t rb = COO_NONE, ra = COO_NONE, ca = 0;
  T va = 0;
  if (i0 < n) { // the arrays' slack covers the last lane's vectors
    const u32x4 rv = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(cr + i0));
    const u32x4 cw = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(cc + i0));
    T w[4];
    if constexpr (sizeof(T) == 4) {
      const f32x4 f = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(cv + i0));
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) w[j] = f[j];
    } else {
      const f64x2 f = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(cv + i0));
      const f64x2 g = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(cv + i0) + 1);
      w[0] = f[0];
      w[1] = f[1];
      w[2] = g[0];
      w[3] = g[1];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; j++)
      if (i0 + j < n) {
        r[j] = rv[j];
        c[j] = cw[j];
        v[j] = w[j];
      }
  }
  if constexpr (OWNER) {
    if (lane < ahead && ia < n) {
      ra = cr[ia];
      ca = cc[ia];
      va = cv[ia];
    }
    if (lane == 0 && w0) rb = cr[w0 - 1];
  }
  T xv[4];
#pragma unroll
  for (uint32_t j = 0; j < 4; j++) xv[j] = x[c[j]]; // entries past n: x[0], not used
  T pv[4];
#pragma unroll
  for (uint32_t j = 0; j < 4; j++) pv[j] = r[j] != COO_NONE ? v[j] * xv[j] : (T)0;
  const uint32_t last = __shfl(r[3], 63, 64);     // row of the span's last entry
  T pa = 0;
  if constexpr (OWNER) {
    if (ra == last && ra != COO_NONE) pa = va * x[ca];
  }
  // the lane's runs: the first (head), those inside, the last (tail)
  T head = pv[0], tail = pv[0];
  bool single = true;
  const uint32_t left = __shfl_up(r[3], 1, 64);
  const uint32_t first = __shfl(r[0], 0, 64);
  // OWNER: the span's first row began before it, and belongs to an earlier wave
  const bool foreign = OWNER && w0 != 0 && __shfl(rb, 0, 64) == first;
  auto put = [&](uint32_t row, T sum) {
    if constexpr (OWNER) {
      if (!(foreign && row == first)) y[row] = sum;
    } else {
      unsafeAtomicAdd(y + row, sum);
    }
  };
#pragma unroll
  for (uint32_t j = 1; j < 4; j++) {
    if (r[j] != r[j - 1]) {
      if (single)
        head = tail;
      else
        put(r[j - 1], tail);
      single = false;
      tail = pv[j];
    } else {
      tail = tail + pv[j];
    }
  }
  // run sums up to the end of each lane: a lane of one row that goes on from
  // the lane before takes that one's sum along
  T scan = tail;
  bool joined = single && lane > 0 && left == r[0];
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const T up = __shfl_up(scan, d, 64);
    const bool jup = __shfl_up((int)joined, d, 64) != 0;
    if (joined && lane >= d) {
      scan = up + scan;
      joined = jup;
    }
    if (!__any(joined && lane >= 2 * d)) break; // no run reaches further back
  }
  const T before = __shfl_up(scan, 1, 64);
  const uint32_t right = __shfl_down(r[0], 1, 64);
  const bool carries = lane > 0 && left == r[0]; // the head began in an earlier lane
  if (r[0] != COO_NONE) {
    if (!single) put(r[0], carries ? before + head : head);
    // the tail ends here unless the next lane goes on with it
    if (lane < 63 ? right != r[3] : !OWNER) {
      if (r[3] != COO_NONE) put(r[3], scan);
    }
  }
  if constexpr (OWNER) {
    if (last != COO_NONE) { // a full span: its last row may go on
      const bool mine = !(foreign && last == first);
      if (mine) { // uniform
        const T more = group_reduce<64>(pa);
        const T sum = __shfl(scan, 63, 64);
        if (lane == 0) y[last] = sum + more;
      }
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_coo(uint64_t n, const uint32_t *__restrict__ cr,
                                             const uint32_t *__restrict__ cc,
                                             const T *__restrict__ cv, const T *__restrict__ x,
                                             T *__restrict__ y)
{
  const uint64_t waves = (uint64_t)gridDim.x * 4u;
  uint64_t w = (uint64_t)blockIdx.x * 4u + (threadIdx.x >> 6);
  for (; w * COO_SPAN < n; w += waves) coo_span<T, false>(w * COO_SPAN, n, 0, cr, cc, cv, x, y);
}

// Owner form: workgroups [0, eblocks) take the entries, the others 256 rows
// each and store the zeros of empty ones.  eblocks and ahead share a word (n is
// below 2^32: 22 and 6 bits), which keeps the arguments in 64 bytes (past them
// the smallest calls took 0.13 us more).
template <typename T>
__global__ __launch_bounds__(256) void k_coo_owner(uint64_t n, uint32_t rows, uint32_t eblocks_ahead,
                                                   const uint32_t *__restrict__ rp, const uint32_t *__restrict__ cr,
                                                   const uint32_t *__restrict__ cc, const T *__restrict__ cv,
                                                   const T *__restrict__ x, T *__restrict__ y)
{
  const uint32_t eblocks = eblocks_ahead / COO_AHEAD, ahead = eblocks_ahead % COO_AHEAD;
  if (blockIdx.x >= eblocks) {
    const uint64_t r = (uint64_t)(blockIdx.x - eblocks) * 256u + threadIdx.x;
    if (r < rows && rp[r] == rp[r + 1]) y[r] = (T)0;
    return;
  }
  const uint64_t w = (uint64_t)xcd_block(blockIdx.x, eblocks) * 4u + (threadIdx.x >> 6);
  if (w * COO_SPAN < n) coo_span<T, true>(w * COO_SPAN, n, ahead, cr, cc, cv, x, y);
}

// Fused hybrid (gpu_matrix_multiplier.cu:969-1002): workgroups [0, ell_blocks)
// run ELL rows with atomic adds, the rest run the COO tail.  y must be zero.
template <typename T>
__global__ __launch_bounds__(256) void k_hyb_atomic(uint32_t rows, uint32_t w,
                                                    const uint32_t *__restrict__ ec,
                                                    const T *__restrict__ ev, uint64_t ncoo,
                                                    const uint32_t *__restrict__ cr,
                                                    const uint32_t *__restrict__ cc,
                                                    const T *__restrict__ cv,
                                                    const T *__restrict__ x, T *__restrict__ y,
                                                    uint32_t ell_blocks)
{
  const uint32_t b = blockIdx.x;
  if (b < ell_blocks) {
    const uint32_t r = b * 256u + threadIdx.x;
    if (r < rows) ell_row<T, true>(r, rows, w, ec, ev, x, y);
    return;
  }
  const uint64_t waves = (uint64_t)(gridDim.x - ell_blocks) * 4u;
  uint64_t wv = (uint64_t)(b - ell_blocks) * 4u + (threadIdx.x >> 6);
  for (; wv * COO_SPAN < ncoo; wv += waves) coo_span<T, false>(wv * COO_SPAN, ncoo, 0, cr, cc, cv, x, y);
}

// ---------------------------------------------------------------------------
// SCOO (scoo_spmv.cu:46-129): one workgroup per slice of slice_size rows.
// Products are added with LDS atomics (ds_add) into acc[row][lane], lane =
// thread % lane_size, then each row's lanes are summed in order.  FP32
// values accumulate in double (A) when acc[slice_size][lane_size] fits in
// LDS that way: the float product is exact in double, and gfx950's
// ds_add_f64 sustains several times the lane rate of ds_add_f32.
// ---------------------------------------------------------------------------
template <typename T, typename A>
__global__ void k_scoo(uint32_t rows, uint32_t ss, uint32_t L, const uint32_t *__restrict__ cr,
                       const uint32_t *__restrict__ cc, const T *__restrict__ cv,
                       const uint32_t *__restrict__ sp, const T *__restrict__ x,
                       T *__restrict__ y)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  A *acc = reinterpret_cast<A *>(smem_raw);
  const uint32_t s = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t r0 = s * ss;
  const uint32_t lim = min(ss, rows - r0);
  const uint32_t bt = blockDim.x, tid = threadIdx.x;
  for (uint32_t i = tid; i < lim * L; i += bt) acc[i] = (A)0;
  __syncthreads();
  const uint32_t b = sp[s], e = sp[s + 1];
  const uint32_t lane = tid & (L - 1u);
  uint32_t i = b + tid;
  for (; i + 3 * bt < e; i += 4 * bt) {
    uint32_t lr[4], c[4];
    T v[4], xv[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      lr[k] = ldg_stream(cr + i + k * bt) - r0;
      c[k] = ldg_stream(cc + i + k * bt);
      v[k] = ldg_stream(cv + i + k * bt);
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) xv[k] = x[c[k]];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++)
      if (lr[k] < lim) atomicAdd(acc + lr[k] * L + lane, (A)v[k] * (A)xv[k]);
  }
  for (; i < e; i += bt) {
    const uint32_t lr = ldg_stream(cr + i) - r0;
    const A p = (A)ldg_stream(cv + i) * (A)x[ldg_stream(cc + i)];
    if (lr < lim) atomicAdd(acc + lr * L + lane, p);
  }
  __syncthreads();
  for (uint32_t lr = tid; lr < lim; lr += bt) {
    A d = 0;
    for (uint32_t l = 0; l < L; l++) d = d + acc[lr * L + l];
    y[r0 + lr] = (T)d;
  }
}

// ---------------------------------------------------------------------------
// Column-sorted SCOO: one workgroup per work item.  The item's slice rows
// accumulate in LDS in double for either value type: a product of two floats
// is exact in double, and on gfx950 ds_add_f64 sustains about 7x the lane
// rate of ds_add_f32 (2.3 against 0.33 lanes per clock per CU with random
// addresses), the rate that bounds this kernel.  Its entries come in column order, so the x
// reads sweep one column range and consecutive lanes share x lines.  Each
// aligned block of 256 positions inside an item is stored word-interleaved:
// a lane's 16-byte load brings positions l, 64 + l, 128 + l and 192 + l, so
// every gather instruction of a wave covers 64 consecutive sorted columns
// (a few x lines) instead of 256 (several times as many L1 lines).  Two
// words per lane are in flight; the unaligned head and tail go one entry
// per lane, in position order.  A slice's
// single item writes y; several write partial slots that k_scoo_cs_finish
// adds in slot order.  Long-row slices work the same way, their local rows
// mapped through long_rows; ordinary slices skip the long rows.  Each y entry
// is written once, with no global atomics (the order of the LDS additions
// still varies from run to run).
// ---------------------------------------------------------------------------
// entry word: (column - item base) << rbits | local row
__device__ __forceinline__ void cs_decode(uint32_t w, uint32_t cbase, uint32_t rbits, uint32_t &c, uint32_t &lr)
{
  c = cbase + (w >> rbits);
  lr = w & ((1u << rbits) - 1u);
}

__device__ __forceinline__ bool cs_is_long(const uint32_t *__restrict__ mask, uint32_t row)
{
  return mask && ((mask[row >> 5] >> (row & 31u)) & 1u);
}

// Stored values of a column-sorted plan: the vector type T itself (DT < 0)
// or 16-bit BF16 / FP16 (DT = MFP_BF16 / MFP_F16, with T = float).  Every
// product is formed in double, exactly: a float, BF16 or FP16 value times a
// float x needs at most 48 significant bits.
template <typename T, int DT>
struct cs_values {
  using V = typename std::conditional<(DT < 0), T, uint16_t>::type;
  __device__ __forceinline__ static double one(const V *__restrict__ ev, uint32_t i)
  {
    if constexpr (DT < 0)
      return (double)ldg_stream(ev + i);
    else
      return (double)lp_val<DT>(ldg_stream(ev + i));
  }
  // the four values of 16-byte entry word g
  __device__ __forceinline__ static void word(const V *__restrict__ ev, uint32_t g, double (&v)[4])
  {
    if constexpr (DT >= 0) {
      const u32x2 h = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(ev) + g);
      v[0] = (double)lp_val<DT>((uint16_t)(h[0] & 0xFFFFu));
      v[1] = (double)lp_val<DT>((uint16_t)(h[0] >> 16));
      v[2] = (double)lp_val<DT>((uint16_t)(h[1] & 0xFFFFu));
      v[3] = (double)lp_val<DT>((uint16_t)(h[1] >> 16));
    } else if constexpr (sizeof(T) == 4) {
      const f32x4 f = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(ev) + g);
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) v[j] = (double)f[j];
    } else {
      // FP64: slots 0, 1 of the block's 64 words, then slots 2, 3 (word g
      // is word g % 64 of block g / 64)
      const f64x2 *p = reinterpret_cast<const f64x2 *>(ev) + (g >> 6) * 128u + (g & 63u);
      const f64x2 d0 = __builtin_nontemporal_load(p);
      const f64x2 d1 = __builtin_nontemporal_load(p + 64);
      v[0] = d0[0];
      v[1] = d0[1];
      v[2] = d1[0];
      v[3] = d1[1];
    }
  }
};

template <typename T, int DT>
__global__ void k_scoo_cs(uint32_t run, uint32_t rows, uint32_t R, uint32_t rbits, uint32_t S_reg, uint32_t NL,
                          const uint4 *__restrict__ items, const uint32_t *__restrict__ ibase,
                          const typename cs_values<T, DT>::V *__restrict__ ev, const uint32_t *__restrict__ ec,
                          const T *__restrict__ x, T *__restrict__ y,
                          T *__restrict__ partial, const uint32_t *__restrict__ long_rows,
                          const uint32_t *__restrict__ long_mask)
{
  using CV = cs_values<T, DT>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *acc = reinterpret_cast<double *>(smem_raw);
  const uint32_t item = xcd_runs(blockIdx.x, gridDim.x, run);
  const uint4 it = items[item];
  const uint32_t sl = it.x, e0 = it.y, e1 = it.z, slot = it.w;
  const uint32_t lim = sl < S_reg ? min(R, rows - sl * R) : min(R, NL - (sl - S_reg) * R);
  const uint32_t bt = blockDim.x, tid = threadIdx.x;
  for (uint32_t i = tid; i < lim; i += bt) acc[i] = 0.0;
  __syncthreads();
  const uint32_t cbase = ibase[item];
  // head: up to the first multiple of 256 (positions stored in order)
  const uint32_t ea = (uint32_t)min<uint64_t>(e1, ((uint64_t)e0 + 255u) & ~(uint64_t)255);
  for (uint32_t i = e0 + tid; i < ea; i += bt) {
    uint32_t c, lr;
    cs_decode(ldg_stream(ec + i), cbase, rbits, c, lr);
    atomicAdd(acc + lr, CV::one(ev, i) * (double)x[c]);
  }
  // body: whole blocks of 256 positions, stored so that 16-byte word l of a
  // block holds positions l, 64 + l, 128 + l, 192 + l; two words per lane in
  // flight.  The decode does not depend on which positions a word holds.
  const uint32_t g0 = ea >> 2, g1 = max(g0, (e1 & ~255u) >> 2); // words [g0, g1) lie inside [ea, e1)
  uint32_t g = g0 + tid;
  for (; g + bt < g1; g += 2 * bt) {
    u32x4 w[2];
    double v[2][4];
#pragma unroll
    for (uint32_t k = 0; k < 2; k++) {
      w[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(ec) + g + k * bt);
      CV::word(ev, g + k * bt, v[k]);
    }
    uint32_t c[2][4], lr[2][4];
    T xv[2][4];
#pragma unroll
    for (uint32_t k = 0; k < 2; k++)
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) cs_decode(w[k][j], cbase, rbits, c[k][j], lr[k][j]);
#pragma unroll
    for (uint32_t k = 0; k < 2; k++)
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) xv[k][j] = x[c[k][j]];
#pragma unroll
    for (uint32_t k = 0; k < 2; k++)
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) atomicAdd(acc + lr[k][j], v[k][j] * (double)xv[k][j]);
  }
  for (; g < g1; g += bt) {
    const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(ec) + g);
    double v[4];
    CV::word(ev, g, v);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      uint32_t c, lr;
      cs_decode(w[j], cbase, rbits, c, lr);
      atomicAdd(acc + lr, v[j] * (double)x[c]);
    }
  }
  // tail: entries after the last whole group
  for (uint32_t i = max(ea, g1 << 2) + tid; i < e1; i += bt) {
    uint32_t c, lr;
    cs_decode(ldg_stream(ec + i), cbase, rbits, c, lr);
    atomicAdd(acc + lr, CV::one(ev, i) * (double)x[c]);
  }
  __syncthreads();
  if (slot == CS_DIRECT && sl >= S_reg) {
    const uint32_t *lrows = long_rows + (uint64_t)(sl - S_reg) * R;
    for (uint32_t lr = tid; lr < lim; lr += bt) y[lrows[lr]] = (T)acc[lr];
  } else if (slot == CS_DIRECT) {
    const uint32_t r0 = sl * R;
    for (uint32_t lr = tid; lr < lim; lr += bt)
      if (!cs_is_long(long_mask, r0 + lr)) y[r0 + lr] = (T)acc[lr];
  } else {
    T *o = partial + (uint64_t)slot * R;
    for (uint32_t lr = tid; lr < lim; lr += bt) o[lr] = (T)acc[lr];
  }
}

// four consecutive values p[0..3] (16-byte aligned)
template <typename T>
__device__ __forceinline__ void load4(const T *__restrict__ p, T (&v)[4])
{
  if constexpr (sizeof(T) == 4) {
    const f32x4 a = *reinterpret_cast<const f32x4 *>(p);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) v[j] = a[j];
  } else {
    const f64x2 a = *reinterpret_cast<const f64x2 *>(p);
    const f64x2 b = *reinterpret_cast<const f64x2 *>(p + 2);
    v[0] = a[0];
    v[1] = a[1];
    v[2] = b[0];
    v[3] = b[1];
  }
}

// sum_in_order for four adjacent rows at once: d[j] = p[j] + p[stride + j]
// + ... in slot order, with 16-byte loads (p 16-byte aligned, stride a
// multiple of 4)
template <typename T>
__device__ __forceinline__ void sum4_in_order(const T *__restrict__ p, uint32_t n, uint64_t stride, T (&d)[4])
{
  load4(p, d);
  for (uint32_t k = 1; k < n; k += 4) {
    T q[4][4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) load4(p + (uint64_t)min(k + i, n - 1) * stride, q[i]);
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) d[j] = (k + i < n) ? d[j] + q[i][j] : d[j];
  }
}

// One workgroup per finish block.  Blocks below NFR: 4 CS_FIN_ROWS rows of
// an ordinary slice, four consecutive rows per thread, y[row] = the slice's
// slots added in slot order (long rows skipped).  The others: CS_FIN_LONG rows of a long-row
// slice, a wave per row; lane l adds slots l, l + 64, ... in order and the
// wave's halving tree adds the lanes, into y[long_rows[(slice - S_reg) R + lr]].
template <typename T>
__global__ __launch_bounds__(CS_FIN_ROWS) void k_scoo_cs_finish(uint32_t rows, uint32_t R, uint32_t S_reg,
                                                                uint32_t NL, uint32_t NFR,
                                                                const uint4 *__restrict__ fin,
                                                                const uint32_t *__restrict__ long_rows,
                                                                const uint32_t *__restrict__ long_mask,
                                                                const T *__restrict__ partial, T *__restrict__ y)
{
  const uint4 f = fin[blockIdx.x];
  const uint32_t sl = f.x, slot0 = f.y, n = f.z;
  if (blockIdx.x >= NFR) {
    const uint32_t lr = f.w + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (lr >= min(R, NL - (sl - S_reg) * R)) return; // uniform across the wave
    // the destination row and up to 8 of the lane's slots are loaded together
    const uint32_t dst = long_rows[(uint64_t)(sl - S_reg) * R + lr];
    const uint32_t cnt = lane < n ? (n - lane + 63u) >> 6 : 0u;
    T d = cnt ? sum_in_order(partial + (uint64_t)(slot0 + lane) * R + lr, cnt, (uint64_t)64 * R) : (T)0;
    d = group_reduce<64>(d);
    if (lane == 0) y[dst] = d;
    return;
  }
  const uint32_t lim = min(R, rows - sl * R);
  const uint32_t lr0 = f.w + 4 * threadIdx.x;
  if (lr0 >= lim || threadIdx.x >= CS_FIN_ROWS) return;
  const T *p = partial + (uint64_t)slot0 * R + lr0;
  const uint32_t row0 = sl * R + lr0;
  T d[4];
  uint32_t lm = 0; // bit j: row0 + j is a long row (its y comes from a long-row slice)
  if ((R & 3u) == 0 && lr0 + 4 <= lim) {
    // row0 is a multiple of 4, so its four mask bits share one word
    if (long_mask) lm = (long_mask[row0 >> 5] >> (row0 & 31u)) & 15u;
    sum4_in_order(p, n, R, d);
  } else {
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      d[j] = lr0 + j < lim ? sum_in_order(p + j, n, R) : (T)0;
      lm |= (lr0 + j < lim && cs_is_long(long_mask, row0 + j)) ? 1u << j : 0u;
    }
  }
  if (lm == 0 && lr0 + 4 <= lim && (reinterpret_cast<uintptr_t>(y + row0) & 15u) == 0) {
    if constexpr (sizeof(T) == 4) {
      *reinterpret_cast<f32x4 *>(y + row0) = f32x4{d[0], d[1], d[2], d[3]};
    } else {
      reinterpret_cast<f64x2 *>(y + row0)[0] = f64x2{d[0], d[1]};
      reinterpret_cast<f64x2 *>(y + row0)[1] = f64x2{d[2], d[3]};
    }
    return;
  }
#pragma unroll
  for (uint32_t j = 0; j < 4; j++)
    if (lr0 + j < lim && !((lm >> j) & 1u)) y[row0 + j] = d[j];
}

// ---------------------------------------------------------------------------
// Column-sorted SCOO SpMM, Y = A X for KV columns (X cols x KV, Y rows x KV,
// row-major): the SpMV kernel above with KV accumulators per slice row
// (acc[column][row], doubles, R KV 8 bytes of LDS: lanes adding one column
// for random rows then spread over the banks, where acc[row][column] would
// put them KV doubles apart) and one X row (KV values, 16-byte loads) per
// entry.  Partial slots hold R KV values, row-major like Y.
// ---------------------------------------------------------------------------
template <typename T, int KV>
__global__ void k_scoo_cs_k(uint32_t run, uint32_t rows, uint32_t R, uint32_t rbits, uint32_t S_reg, uint32_t NL,
                            const uint4 *__restrict__ items, const uint32_t *__restrict__ ibase,
                            const T *__restrict__ ev, const uint32_t *__restrict__ ec, const T *__restrict__ X,
                            T *__restrict__ Y, T *__restrict__ partial, const uint32_t *__restrict__ long_rows,
                            const uint32_t *__restrict__ long_mask)
{
  using CV = cs_values<T, -1>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *acc = reinterpret_cast<double *>(smem_raw);
  const uint32_t item = xcd_runs(blockIdx.x, gridDim.x, run);
  const uint4 it = items[item];
  const uint32_t sl = it.x, e0 = it.y, e1 = it.z, slot = it.w;
  const uint32_t lim = sl < S_reg ? min(R, rows - sl * R) : min(R, NL - (sl - S_reg) * R);
  const uint32_t bt = blockDim.x, tid = threadIdx.x;
  for (uint32_t i = tid; i < R * KV; i += bt) acc[i] = 0.0;
  __syncthreads();
  const uint32_t cbase = ibase[item];
  auto add_row = [&](uint32_t c, uint32_t lr, double v) {
    T xr[KV];
    load_row<T, KV>(X + (uint64_t)c * KV, xr);
#pragma unroll
    for (int j = 0; j < KV; j++) atomicAdd(acc + j * R + lr, v * (double)xr[j]);
  };
  const uint32_t ea = (uint32_t)min<uint64_t>(e1, ((uint64_t)e0 + 255u) & ~(uint64_t)255);
  for (uint32_t i = e0 + tid; i < ea; i += bt) {
    uint32_t c, lr;
    cs_decode(ldg_stream(ec + i), cbase, rbits, c, lr);
    add_row(c, lr, CV::one(ev, i));
  }
  // body: one 16-byte entry word (four entries) per lane per step
  const uint32_t g0 = ea >> 2, g1 = max(g0, (e1 & ~255u) >> 2);
  for (uint32_t g = g0 + tid; g < g1; g += bt) {
    const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(ec) + g);
    double v[4];
    CV::word(ev, g, v);
    uint32_t c[4], lr[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) cs_decode(w[j], cbase, rbits, c[j], lr[j]);
    T xr[4][KV];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) load_row<T, KV>(X + (uint64_t)c[j] * KV, xr[j]);
#pragma unroll
    for (uint32_t j = 0; j < 4; j++)
#pragma unroll
      for (int q = 0; q < KV; q++) atomicAdd(acc + q * R + lr[j], v[j] * (double)xr[j][q]);
  }
  for (uint32_t i = max(ea, g1 << 2) + tid; i < e1; i += bt) {
    uint32_t c, lr;
    cs_decode(ldg_stream(ec + i), cbase, rbits, c, lr);
    add_row(c, lr, CV::one(ev, i));
  }
  __syncthreads();
  if (slot == CS_DIRECT && sl >= S_reg) {
    const uint32_t *lrows = long_rows + (uint64_t)(sl - S_reg) * R;
    for (uint32_t i = tid; i < lim * KV; i += bt)
      Y[(uint64_t)lrows[i / KV] * KV + i % KV] = (T)acc[(i % KV) * R + i / KV];
  } else if (slot == CS_DIRECT) {
    const uint64_t r0 = (uint64_t)sl * R;
    for (uint32_t i = tid; i < lim * KV; i += bt)
      if (!cs_is_long(long_mask, (uint32_t)(r0 + i / KV))) Y[r0 * KV + i] = (T)acc[(i % KV) * R + i / KV];
  } else {
    T *o = partial + (uint64_t)slot * R * KV;
    for (uint32_t i = tid; i < lim * KV; i += bt) o[i] = (T)acc[(i % KV) * R + i / KV];
  }
}

// The SpMM finish: as k_scoo_cs_finish, over (row, column) pairs; each
// pair's slots are added in slot order.
template <typename T>
__global__ __launch_bounds__(CS_FIN_ROWS) void k_scoo_cs_finish_k(uint32_t rows, uint32_t R, uint32_t KV,
                                                                  uint32_t S_reg, uint32_t NL, uint32_t NFR,
                                                                  const uint4 *__restrict__ fin,
                                                                  const uint32_t *__restrict__ long_rows,
                                                                  const uint32_t *__restrict__ long_mask,
                                                                  const T *__restrict__ partial,
                                                                  T *__restrict__ Y)
{
  const uint4 f = fin[blockIdx.x];
  const uint32_t sl = f.x, slot0 = f.y, n = f.z;
  const uint64_t stride = (uint64_t)R * KV;
  const T *p = partial + (uint64_t)slot0 * stride;
  if (blockIdx.x >= NFR) {
    const uint32_t lim = min(R, NL - (sl - S_reg) * R);
    for (uint32_t i = threadIdx.x; i < CS_FIN_LONG * KV; i += CS_FIN_ROWS) {
      const uint32_t lr = f.w + i / KV, j = i % KV;
      if (lr < lim) Y[(uint64_t)long_rows[(uint64_t)(sl - S_reg) * R + lr] * KV + j] = sum_in_order(p + (uint64_t)lr * KV + j, n, stride);
    }
    return;
  }
  const uint32_t lim = min(R, rows - sl * R);
  for (uint32_t i = threadIdx.x; i < 4 * CS_FIN_ROWS * KV; i += CS_FIN_ROWS) {
    const uint32_t lr = f.w + i / KV, j = i % KV;
    const uint32_t row = sl * R + lr;
    if (lr < lim && !cs_is_long(long_mask, row))
      Y[(uint64_t)row * KV + j] = sum_in_order(p + (uint64_t)lr * KV + j, n, stride);
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static int launched()
{
  mark_kernel_end();
  return hipGetLastError() == hipSuccess ? MFP_OK : (set_error("kernel launch failed"), MFP_ERR_HIP);
}

// launch status of a kernel launched with its own start / stop events
static int launched_timed()
{
  return hipGetLastError() == hipSuccess ? MFP_OK : (set_error("kernel launch failed"), MFP_ERR_HIP);
}

// Launch a kernel and check the launch.  Under mfp_plan_kernel_times the
// kernel records its own start and end (hipExtLaunchKernelGGL events);
// otherwise it is a plain launch followed by the usual mark.
template <typename... P, typename... A>
static int launch_k(void (*kernel)(P...), dim3 grid, dim3 block, uint32_t lds, hipStream_t s, A... args)
{
  hipEvent_t e0, e1;
  if (mark_kernel_events(&e0, &e1)) {
    hipExtLaunchKernelGGL(kernel, grid, block, lds, s, e0, e1, 0u, static_cast<P>(args)...);
    return launched_timed();
  }
  hipLaunchKernelGGL(kernel, grid, block, lds, s, static_cast<P>(args)...);
  return launched();
}

// Rows per workgroup of k_csr_vector_lds, 0 where k_csr_vector serves the
// matrix.  The LDS form for rows of up to CAP / 8 entries on average (256 FP32,
// 128 FP64: enough rows per chunk for every group of lanes) and for rows of
// 2 CAP or more (whole chunks); between them a chunk holds one to seven
// rows and most groups idle: rows of about 1,200 took 25 us here against
// 27 to 301 from LDS, 64 to 2 lanes.
// A small matrix is a chain of latencies in either form, and the LDS form's is
// longer.  From 8 MB of entries it is the faster one (lanes from the mean, FP32
// row by row -> LDS: 800k entries in rows of 6, 34, 100 6.8 -> 7.6, 6.8 -> 7.2,
// 4.6 -> 4.8 us, 1.6M 12.5 -> 13.1, 12.5 -> 11.8, 9.8 -> 8.6; FP64 400k 4.9 ->
// 5.3, 5.5 -> 5.3, 3.7 -> 4.0, 800k 9.0 -> 8.4, 9.1 -> 8.0, 6.8 -> 5.6), and
// earlier where lanes idle (FP32 rows of 6 by 64 lanes, 33k and 67k rows: 5.7 ->
// 6.7, 11.0 -> 10.6 us) or a row is several waits of its lanes (rows of 34 by 4
// lanes, 135k, 200k, 400k entries: 3.9 -> 4.0, 4.2 -> 4.0, 6.0 -> 4.4 us).
uint32_t csr_vector_rows(int dtype, uint32_t lanes, uint32_t rows, uint64_t nnz)
{
  if (rows == 0) return 0;
  const uint32_t cap = dtype == MFP_F32 ? cvl<float>::CAP : cvl<double>::CAP;
  const uint64_t vs = dtype_size(dtype);
  const double mean = (double)nnz / rows;
  if (mean > cap / 8 && mean < 2.0 * cap) return 0;
  if (nnz * (4 + vs) < 8u << 20 && (uint64_t)rows * lanes * vs < 16u << 20 && !(nnz >= 1u << 18 && mean >= 4.0 * lanes))
    return 0;
  // rows that fill 85% of a chunk on average, fewer where that would leave
  // a CU with less than two workgroups
  const uint32_t fit = (uint32_t)std::min(256.0, std::max(1.0, 0.85 * cap / std::max(mean, 1.0)));
  return std::max(1u, std::min(fit, ceil_div_u32(rows, 2u * (uint32_t)std::max(1, props().cu_count))));
}

// Lists the blocks of RB rows whose rows would keep their one workgroup busy
// for longer than `limit` and than their own lanes would take side by side.
// Times in ns: a chunk waits 800, gathers at 0.85 per entry and then takes 8
// per step of its longest row's lanes (a row that shares a chunk: its part of
// all that); row by row, a row's lanes wait 570 per CVL_REST entries of each.
// A wave per block.
template <typename T>
__global__ __launch_bounds__(256) void k_csr_vector_blocks(uint32_t rows, uint32_t RB, uint32_t nblocks, float lanes,
                                                           float limit, const uint32_t *__restrict__ rp,
                                                           uint32_t *__restrict__ list, uint32_t *__restrict__ mask,
                                                           uint32_t *__restrict__ count)
{
  constexpr float CAP = cvl<T>::CAP, CHUNK = cvl<T>::CHUNK;
  const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (w >= nblocks) return; // the whole wave
  const uint32_t r0 = w * RB, nr = min(RB, rows - r0);
  if (rp[r0 + nr] - rp[r0] <= cvl<T>::CAP - cvl<T>::N) return;
  float chunks = 0, longest = 0;
  for (uint32_t r = lane; r < nr; r += 64) {
    const float len = (float)(rp[r0 + r + 1] - rp[r0 + r]);
    longest = fmaxf(longest, len);
    if (len > CAP)
      chunks += ceilf(len / CHUNK) * (800.0f + 0.85f * CHUNK + 8.0f * CHUNK / lanes);
    else
      chunks += (960.0f / CAP + 0.85f) * len + 8.0f * fmaxf(len * len / (lanes * CAP), fmaxf(lanes, len) / 256.0f);
  }
  chunks = group_reduce<64>(chunks);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) longest = fmaxf(longest, __shfl_xor(longest, d, 64));
  chunks += 800.0f;
  if (lane == 0 && chunks > limit && chunks > 2500.0f + 570.0f * longest / (CVL_REST * lanes)) {
    atomicOr(&mask[w >> 5], 1u << (w & 31u));
    list[atomicAdd(count, 1u)] = w;
  }
}

// A workgroup sums its block's rows chunk after chunk.  Where long rows lie
// side by side (rows sorted by length, a dense stretch) that is a chain of
// hundreds of chunks on one CU, while their own lanes would work on all of them
// at once: such blocks are listed and summed row by row, in the same launch, a
// wave per workgroup while they are few.  300,007 rows of 6 with 256 rows of
// 1,500 among them, FP32, 8 lanes: row by row 68 us, all from LDS 3,214,
// listed 30 (4 lanes 157, 5,884, 59; FP64 77, 683, 32); 1M power-law rows
// sorted by length 845, 6,610, 780 (FP64 1,170, 7,803, 560), unsorted 341, 175,
// 176.  One row of 9,000 entries among 47,000 of 34, 64 lanes, is the case that
// stays behind the row-by-row form: 15.6 against 18.6 us.
int csr_vector_layout_build(int dtype, uint32_t lanes, uint32_t rows, uint64_t nnz, uint32_t longest,
                            const uint32_t *rp, csr_vector_layout *out, hipStream_t s)
{
  *out = csr_vector_layout{};
  out->rb = csr_vector_rows(dtype, lanes, rows, nnz);
  const bool f32 = dtype == MFP_F32;
  const uint32_t cap = f32 ? cvl<float>::CAP : cvl<double>::CAP;
  if (out->rb <= 1 || (uint64_t)out->rb * longest <= 2 * cap) return MFP_OK; // no block is that long
  // a quarter of what the whole product takes at least (1.5 TB/s, a launch)
  const float limit = 0.25f * std::max(4000.0f, (float)nnz * (float)(4 + dtype_size(dtype)) / 1500.0f);
  const uint32_t nb = ceil_div_u32(rows, out->rb), words = (nb + 31) / 32;
  // mask, count, list
  MFP_CHECK(dmalloc((void **)&out->mask, ((uint64_t)words + 1 + nb) * 4));
  uint32_t *count = out->mask + words;
  out->list = count + 1;
  int st = fill_u32(out->mask, 0, (uint64_t)words + 1, s);
  if (st == MFP_OK) {
    const auto kern = f32 ? k_csr_vector_blocks<float> : k_csr_vector_blocks<double>;
    kern<<<ceil_div_u32(nb, 4), 256, 0, s>>>(rows, out->rb, nb, (float)lanes, limit, rp, out->list, out->mask, count);
    st = launched();
  }
  if (st == MFP_OK && (hipMemcpyAsync(&out->count, count, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
                       hipStreamSynchronize(s) != hipSuccess)) {
    set_error("CSR-vector: blocks of long rows");
    st = MFP_ERR_HIP;
  }
  const uint64_t per = (out->rb * (uint64_t)lanes + 255) / 256;
  if (st != MFP_OK || out->count == 0 || !grid_fits(out->count * per + nb + 8, 256)) csr_vector_layout_free(out);
  return st;
}

void csr_vector_layout_free(csr_vector_layout *l)
{
  if (l->mask) {
    const beside_capture mode;
    dfree(l->mask);
  }
  l->mask = l->list = nullptr;
  l->count = 0;
}

template <typename T, int G>
static int csr_vector_g(uint32_t rows, const csr_vector_layout &l, const uint32_t *rp, const uint32_t *ci, const T *a,
                        const T *x, T *y, hipStream_t s)
{
  const dim3 b(256);
  if (l.rb) {
    // few listed blocks spread over the CUs, a wave per workgroup
    uint32_t lists = 64;
    while (lists < 256 && l.count * ((l.rb * G + lists - 1) / lists) > 4u * (uint32_t)std::max(1, props().cu_count))
      lists *= 2;
    const uint32_t extra = (l.count * ((l.rb * G + lists - 1) / lists) + 7u) & ~7u;
    return launch_k(k_csr_vector_lds<T, G>, dim3(extra + ceil_div_u32(rows, l.rb)), b, 0, s, rows, l.rb, extra, lists,
                    l.count, l.list, l.mask, rp, ci, a, x, y);
  }
  const uint32_t grid = ceil_div_u32((uint64_t)rows * G, 256);
  return launch_k(k_csr_vector<T, G>, dim3(grid), b, 0, s, rows, rp, ci, a, x, y);
}

template <typename T>
static int csr_vector_t(uint32_t lanes, uint32_t rows, const csr_vector_layout &l, const uint32_t *rp,
                        const uint32_t *ci, const T *a, const T *x, T *y, hipStream_t s)
{
  switch (lanes) {
  case 2: return csr_vector_g<T, 2>(rows, l, rp, ci, a, x, y, s);
  case 4: return csr_vector_g<T, 4>(rows, l, rp, ci, a, x, y, s);
  case 8: return csr_vector_g<T, 8>(rows, l, rp, ci, a, x, y, s);
  case 16: return csr_vector_g<T, 16>(rows, l, rp, ci, a, x, y, s);
  case 32: return csr_vector_g<T, 32>(rows, l, rp, ci, a, x, y, s);
  case 64: return csr_vector_g<T, 64>(rows, l, rp, ci, a, x, y, s);
  default: set_error("lanes must be a power of two in [2, 64]"); return MFP_ERR_ARG;
  }
}

int launch_csr_scalar(int dtype, uint32_t rows, const uint32_t *rp, const uint32_t *ci,
                      const void *a, const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  const uint32_t grid = ceil_div_u32(rows, 64);
  if (dtype == MFP_F32)
    return launch_k(k_csr_scalar<float>, dim3(grid), dim3(64), 0, s, rows, rp, ci, (const float *)a,
                    (const float *)x, (float *)y);
  return launch_k(k_csr_scalar<double>, dim3(grid), dim3(64), 0, s, rows, rp, ci, (const double *)a,
                  (const double *)x, (double *)y);
}

int launch_csr_vector(int dtype, uint32_t lanes, uint32_t rows, const csr_vector_layout &l, const uint32_t *rp,
                      const uint32_t *ci, const void *a, const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  if (dtype == MFP_F32)
    return csr_vector_t<float>(lanes, rows, l, rp, ci, (const float *)a, (const float *)x, (float *)y, s);
  return csr_vector_t<double>(lanes, rows, l, rp, ci, (const double *)a, (const double *)x, (double *)y, s);
}

// Vectors a lane may need for a block of up to W elements at any alignment.
uint32_t adaptive_vectors_per_lane(int dtype, uint32_t W)
{
  const uint32_t N = dtype == MFP_F32 ? 4 : 2;
  const uint32_t maxvec = (W + 2 * N - 2) / N;
  uint32_t k = (maxvec + AD_T - 1) / AD_T;
  uint32_t p = 1;
  while (p < k) p <<= 1;
  return p;
}

template <typename T, uint32_t K>
static int adaptive_launch_k(const adaptive_args &g, const T *a, const T *x, T *y, hipStream_t s, uint32_t gap,
                             size_t lds, uint32_t items, uint32_t nchunks_pad)
{
  const auto fn = g.batch ? k_csr_adaptive<T, K, true> : k_csr_adaptive<T, K, false>;
  if (lds > 65536)
    MFP_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  return launch_k(fn, dim3(items), dim3(AD_T), (uint32_t)lds, s, g.rp, g.ci, a, x, y, g.blocks, g.nnz_per_wg,
                  g.long_row, g.chunks, g.nchunks, nchunks_pad, g.chunk, gap, (T *)g.partials);
}

// Dynamic LDS of k_csr_adaptive: the staged products, then the row starts.
template <typename T>
static size_t adaptive_lds_bytes(uint32_t W, uint32_t gap)
{
  return adaptive_products<T>(W, gap) + ((size_t)W + 2) * 4;
}

// The gaps between the products, unless a CU would hold fewer workgroups with
// them: us with and without, 27-point 100^3, FP64 W = 1,800, 2,800, 4,000 73.0 and
// 68.3, 91.8 and 77.7, 107.5 and 81.3, FP32 W = 2,600, 4,700, 6,300 61.3 and 57.2,
// 79.7 and 68.4, 100.2 and 73.8; where as many fit (FP32 W = 8,000) 92.7 and 104.8.
template <typename T>
static uint32_t adaptive_gap(uint32_t W)
{
  const size_t lds = 160u << 10, own = 2 * AD_T * sizeof(T) + 64; // sv, wsum, wsteps
  constexpr uint32_t gap = sizeof(T) == 4 ? 3 : 2;
  const auto groups = [&](uint32_t q) { return std::min<size_t>(8, lds / (adaptive_lds_bytes<T>(W, q) + own)); };
  return groups(gap) < groups(ADAPTIVE_NO_GAP) ? ADAPTIVE_NO_GAP : gap;
}

// Workgroups of one launch: their lanes are numbered in 32 bits.  Blocks of one
// entry are that many from 16.7M entries on.
constexpr uint32_t ADAPTIVE_GRID = (1u << 24) - 8;

template <typename T>
static int adaptive_t(const adaptive_args &g, const T *a, const T *x, T *y, hipStream_t s)
{
  // chunk items first; padded to a multiple of 8 so block ids keep their XCD
  const uint32_t nchunks_pad = (g.nchunks + 7u) & ~7u;
  const uint32_t items = g.nblocks ? g.nblocks + nchunks_pad : nchunks_pad;
  const uint32_t gap = adaptive_gap<T>(g.nnz_per_wg);
  const size_t lds = adaptive_lds_bytes<T>(g.nnz_per_wg, gap);
  const uint32_t K = adaptive_vectors_per_lane(sizeof(T) == 4 ? MFP_F32 : MFP_F64, g.nnz_per_wg);
  adaptive_args part = g;
  uint32_t pad = nchunks_pad;
  for (uint32_t left = items; left;) {
    const uint32_t n = pad < ADAPTIVE_GRID ? std::min(left, ADAPTIVE_GRID) : left;
    int st;
    switch (K) {
    case 1: st = adaptive_launch_k<T, 1>(part, a, x, y, s, gap, lds, n, pad); break;
    case 2: st = adaptive_launch_k<T, 2>(part, a, x, y, s, gap, lds, n, pad); break;
    case 4: st = adaptive_launch_k<T, 4>(part, a, x, y, s, gap, lds, n, pad); break;
    case 8: st = adaptive_launch_k<T, 8>(part, a, x, y, s, gap, lds, n, pad); break;
    case 16: st = adaptive_launch_k<T, 16>(part, a, x, y, s, gap, lds, n, pad); break;
    default: set_error("nnz_per_wg too large"); return MFP_ERR_ARG;
    }
    MFP_CHECK(st);
    left -= n;
    part.blocks += n - pad;
    part.nchunks = pad = 0;
  }
  if (g.nchunks)
    MFP_CHECK(launch_k(k_adaptive_finish<T>, dim3(ceil_div_u32(g.nchunks, 256)), dim3(256), 0, s, g.chunks,
                       g.nchunks, (const T *)g.partials, y));
  return MFP_OK;
}

int launch_csr_adaptive(int dtype, const adaptive_args &g, const void *a, const void *x, void *y,
                        hipStream_t s)
{
  if (dtype == MFP_F32) return adaptive_t<float>(g, (const float *)a, (const float *)x, (float *)y, s);
  return adaptive_t<double>(g, (const double *)a, (const double *)x, (double *)y, s);
}

int launch_ell_pk(int dtype, uint32_t rows, uint32_t w, uint32_t w4, const uint32_t *base, const void *val,
                  const uint16_t *off, const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  const dim3 grid(ceil_div_u32(rows, 256));
  if (dtype == MFP_F32)
    return launch_k(k_ell_pk<float>, grid, dim3(256), 0, s, rows, w, w4, base, (const f32x4 *)val,
                    (const pk_u16x4 *)off, (const float *)x, (float *)y);
  return launch_k(k_ell_pk<double>, grid, dim3(256), 0, s, rows, w, w4, base, (const f64x2 *)val,
                  (const pk_u16x4 *)off, (const double *)x, (double *)y);
}

int ell_pk_build(int dtype, uint32_t rows, uint32_t stride, const uint32_t *rp, const uint32_t *ci, const void *a,
                 uint32_t w4, const uint32_t *base, void *val, uint16_t *off, hipStream_t s)
{
  if (stride == 0) return MFP_OK;
  const uint32_t g = ceil_div_u32(stride, 256);
  if (dtype == MFP_F32)
    k_ell_pk_build<float><<<g, 256, 0, s>>>(rows, stride, rp, ci, (const float *)a, w4, base, (float *)val, off);
  else
    k_ell_pk_build<double><<<g, 256, 0, s>>>(rows, stride, rp, ci, (const double *)a, w4, base, (double *)val, off);
  return hipGetLastError() == hipSuccess ? MFP_OK : (set_error("packed ELL build failed"), MFP_ERR_HIP);
}

int launch_ell(int dtype, uint32_t rows, uint32_t w, const uint32_t *ec, const void *ev,
               const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  const uint32_t grid = ceil_div_u32(rows, 256);
  if (dtype == MFP_F32)
    return launch_k(k_ell<float>, dim3(grid), dim3(256), 0, s, rows, w, ec, (const float *)ev, (const float *)x,
                    (float *)y);
  return launch_k(k_ell<double>, dim3(grid), dim3(256), 0, s, rows, w, ec, (const double *)ev, (const double *)x,
                  (double *)y);
}

int launch_vec_add(int dtype, uint32_t n, const void *t, void *y, hipStream_t s)
{
  if (n == 0) return MFP_OK;
  const uint32_t grid = ceil_div_u32(n, 256);
  if (dtype == MFP_F32)
    return launch_k(k_vec_add<float>, dim3(grid), dim3(256), 0, s, n, (const float *)t, (float *)y);
  return launch_k(k_vec_add<double>, dim3(grid), dim3(256), 0, s, n, (const double *)t, (double *)y);
}

static uint32_t coo_grid(uint64_t n)
{
  const uint64_t per_block = 4u * COO_SPAN;
  const uint64_t tiles = (n + per_block - 1) / per_block;
  const uint64_t cap = (uint64_t)std::max(1, props().cu_count) * 16u;
  return (uint32_t)std::max<uint64_t>(1, std::min(tiles, cap));
}

int launch_coo_add(int dtype, uint64_t n, const uint32_t *cr, const uint32_t *cc, const void *cv,
                   const void *x, void *y, hipStream_t s)
{
  if (n == 0) return MFP_OK;
  const uint32_t grid = coo_grid(n);
  if (dtype == MFP_F32)
    return launch_k(k_coo<float>, dim3(grid), dim3(256), 0, s, n, cr, cc, (const float *)cv, (const float *)x,
                    (float *)y);
  return launch_k(k_coo<double>, dim3(grid), dim3(256), 0, s, n, cr, cc, (const double *)cv, (const double *)x,
                  (double *)y);
}

bool coo_owner_fits(uint64_t n, uint32_t rows, uint32_t longest_row)
{
  return longest_row <= COO_AHEAD && n < 1ull << 32 && // k_coo_owner's word
         grid_fits((uint64_t)ceil_div_u32(n, 4u * COO_SPAN) + ceil_div_u32(rows, 256), 256);
}

int launch_coo_owner(int dtype, uint32_t rows, uint64_t n, uint32_t longest_row, const uint32_t *rp, const uint32_t *cr,
                     const uint32_t *cc, const void *cv, const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  const uint32_t eb = ceil_div_u32(n, 4u * COO_SPAN), grid = eb + ceil_div_u32(rows, 256);
  const uint32_t word = eb * COO_AHEAD + (longest_row ? longest_row - 1u : 0u);
  if (dtype == MFP_F32)
    return launch_k(k_coo_owner<float>, dim3(grid), dim3(256), 0, s, n, rows, word, rp, cr, cc, (const float *)cv,
                    (const float *)x, (float *)y);
  return launch_k(k_coo_owner<double>, dim3(grid), dim3(256), 0, s, n, rows, word, rp, cr, cc, (const double *)cv,
                  (const double *)x, (double *)y);
}

int launch_hyb_atomic(int dtype, uint32_t rows, uint32_t w, const uint32_t *ec, const void *ev,
                      uint64_t ncoo, const uint32_t *cr, const uint32_t *cc, const void *cv,
                      const void *x, void *y, hipStream_t s)
{
  const uint32_t eb = w ? ceil_div_u32(rows, 256) : 0u;
  const uint32_t cb = ncoo ? coo_grid(ncoo) : 0u;
  if (eb + cb == 0) return MFP_OK;
  if (dtype == MFP_F32)
    return launch_k(k_hyb_atomic<float>, dim3(eb + cb), dim3(256), 0, s, rows, w, ec, (const float *)ev, ncoo, cr,
                    cc, (const float *)cv, (const float *)x, (float *)y, eb);
  return launch_k(k_hyb_atomic<double>, dim3(eb + cb), dim3(256), 0, s, rows, w, ec, (const double *)ev, ncoo, cr,
                  cc, (const double *)cv, (const double *)x, (double *)y, eb);
}

int launch_scoo(int dtype, uint32_t rows, uint32_t ss, uint32_t L, uint32_t threads,
                const uint32_t *cr, const uint32_t *cc, const void *cv, const uint32_t *sp,
                const void *x, void *y, hipStream_t s)
{
  if (rows == 0) return MFP_OK;
  if (ss == 0 || L == 0 || (L & (L - 1)) != 0) {
    set_error("SCOO geometry: slice_size > 0 and a power-of-two lane_size are required");
    return MFP_ERR_ARG;
  }
  if (threads == 0 || threads > 1024 || threads % 64 != 0) {
    set_error("SCOO workgroup size must be a multiple of 64 up to 1024");
    return MFP_ERR_ARG;
  }
  const size_t lds = (size_t)ss * L * dtype_size(dtype);
  if (lds > 160u * 1024u) {
    set_error("SCOO slice_size * lane_size exceeds the 160 KB LDS of a workgroup");
    return MFP_ERR_ARG;
  }
  const uint32_t real = ceil_div_u32(rows, ss);
  auto go = [&](auto kern, size_t bytes, auto tv) -> int {
    using TV = decltype(tv);
    if (bytes > 65536)
      MFP_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return launch_k(kern, dim3(real), dim3(threads), (uint32_t)bytes, s, rows, ss, L, cr, cc, (const TV *)cv, sp,
                    (const TV *)x, (TV *)y);
  };
  if (dtype == MFP_F64)
    MFP_CHECK(go(k_scoo<double, double>, lds, 0.0));
  else if (2 * lds <= 160u * 1024u)
    MFP_CHECK(go(k_scoo<float, double>, 2 * lds, 0.0f));
  else
    MFP_CHECK(go(k_scoo<float, float>, lds, 0.0f));
  return MFP_OK;
}

template <typename T, int DT>
static int scoo_cs_t(uint32_t rows, const scoo_cs_layout &l, uint32_t threads, const void *x, void *y,
                     hipStream_t s)
{
  using V = typename cs_values<T, DT>::V;
  const size_t lds = (size_t)l.R * sizeof(double);
  if (lds > 65536)
    MFP_HIP(hipFuncSetAttribute((const void *)k_scoo_cs<T, DT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  MFP_CHECK(launch_k(k_scoo_cs<T, DT>, dim3(l.NI), dim3(threads), (uint32_t)lds, s, l.run, rows, l.R, l.rbits,
                     l.S_reg, l.NL, l.items, l.base, (const V *)l.ev, l.ec, (const T *)x, (T *)y, (T *)l.partial,
                     l.long_rows, l.long_mask));
  if (l.NF)
    MFP_CHECK(launch_k(k_scoo_cs_finish<T>, dim3(l.NF), dim3(CS_FIN_ROWS), 0, s, rows, l.R, l.S_reg, l.NL, l.NFR,
                       l.fin, l.long_rows, l.long_mask, (const T *)l.partial, (T *)y));
  return MFP_OK;
}

template <typename T, int KV>
static int scoo_cs_k_t(uint32_t rows, const scoo_cs_layout &l, uint32_t threads, const void *X, void *Y,
                       hipStream_t s)
{
  const size_t lds = (size_t)l.R * KV * sizeof(double);
  if (lds > 65536)
    MFP_HIP(hipFuncSetAttribute((const void *)k_scoo_cs_k<T, KV>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  k_scoo_cs_k<T, KV><<<l.NI, threads, lds, s>>>(l.run, rows, l.R, l.rbits, l.S_reg, l.NL, l.items, l.base,
                                                (const T *)l.ev, l.ec, (const T *)X, (T *)Y, (T *)l.partial,
                                                l.long_rows, l.long_mask);
  MFP_CHECK(launched());
  if (l.NF) {
    k_scoo_cs_finish_k<T><<<l.NF, CS_FIN_ROWS, 0, s>>>(rows, l.R, KV, l.S_reg, l.NL, l.NFR, l.fin, l.long_rows,
                                                        l.long_mask, (const T *)l.partial, (T *)Y);
    MFP_CHECK(launched());
  }
  return MFP_OK;
}

int launch_scoo_cs_spmm(int dtype, uint32_t k, uint32_t rows, const scoo_cs_layout &l, uint32_t threads,
                        const void *X, void *Y, hipStream_t s)
{
  if (dtype != MFP_F32 && dtype != MFP_F64) {
    set_error("column-sorted SpMM values must be f32 or f64");
    return MFP_ERR_ARG;
  }
  if (k > l.kmax) {
    set_error("column-sorted SpMM: slice_size * k doubles exceed the 160 KB LDS (use smaller slices)");
    return MFP_ERR_ARG;
  }
  if ((k * dtype_size(dtype)) % 16 == 0 && ((uintptr_t)X % 16) != 0) {
    set_error("X must be 16-byte aligned when its rows are a multiple of 16 bytes");
    return MFP_ERR_ARG;
  }
  if (threads == 0 || threads > 1024 || threads % 64) {
    set_error("SCOO workgroup size must be a multiple of 64 up to 1024");
    return MFP_ERR_ARG;
  }
  if (rows == 0 || l.NI == 0) return MFP_OK;
  const bool f32 = dtype == MFP_F32;
  switch (k) {
  case 2: return f32 ? scoo_cs_k_t<float, 2>(rows, l, threads, X, Y, s) : scoo_cs_k_t<double, 2>(rows, l, threads, X, Y, s);
  case 4: return f32 ? scoo_cs_k_t<float, 4>(rows, l, threads, X, Y, s) : scoo_cs_k_t<double, 4>(rows, l, threads, X, Y, s);
  case 8: return f32 ? scoo_cs_k_t<float, 8>(rows, l, threads, X, Y, s) : scoo_cs_k_t<double, 8>(rows, l, threads, X, Y, s);
  case 16: return f32 ? scoo_cs_k_t<float, 16>(rows, l, threads, X, Y, s) : scoo_cs_k_t<double, 16>(rows, l, threads, X, Y, s);
  }
  set_error("k must be 1, 2, 4, 8 or 16");
  return MFP_ERR_ARG;
}

int launch_scoo_cs(int dtype, uint32_t rows, const scoo_cs_layout &l, uint32_t threads, const void *x, void *y,
                   hipStream_t s)
{
  if (rows == 0 || l.NI == 0) return MFP_OK;
  const size_t lds = (size_t)l.R * sizeof(double);
  if (lds > 163840) {
    set_error("column-sorted SCOO slice exceeds the LDS of a workgroup");
    return MFP_ERR_ARG;
  }
  if (threads == 0 || threads > 1024 || threads % 64) {
    set_error("SCOO workgroup size must be a multiple of 64 up to 1024");
    return MFP_ERR_ARG;
  }
  switch (dtype) {
  case MFP_F32: return scoo_cs_t<float, -1>(rows, l, threads, x, y, s);
  case MFP_F64: return scoo_cs_t<double, -1>(rows, l, threads, x, y, s);
  case MFP_BF16: return scoo_cs_t<float, MFP_BF16>(rows, l, threads, x, y, s);
  case MFP_F16: return scoo_cs_t<float, MFP_F16>(rows, l, threads, x, y, s);
  }
  set_error("column-sorted SCOO: unknown value type");
  return MFP_ERR_ARG;
}

} // namespace mfp
