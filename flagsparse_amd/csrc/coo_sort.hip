// COO entries into row order on the device: a stable radix sort by row that carries the columns
// and values, and the row pointers of row-ordered entries.
//
// Reference behaviour replaced: the lexicographic sorts of spmv_coo.py:153-164 and
// spmm_coo.py:136-180 before a product.  A product needs each row's entries together, not their
// order inside the row, so the sort is by row alone; it is stable, so the result, and the order
// of every sum, is a function of the input.
//
// As a 64-bit key (row * n_cols + col), an argsort and three gathers, that was 11 passes over
// 12-byte pairs whatever the matrix, plus random reads of the entries (measured on MI355X: 330 us
// for 1.65M entries of 150k rows, 240 us for 1.2M of 60k).  Here only the bits that the rows have
// are sorted, up to 9 a pass (two passes to 262,144 rows, three to 134M), 16 bytes an entry.
// A pass is three launches:
//   coo_hist_kernel     digits of each tile of 2048 or 4096 entries -> counts[digit][tile]
//   coo_scan_kernel     a workgroup per digit: exclusive sums over the tiles, the digit's total
//   coo_scatter_kernel  each tile ranks its entries (wave ballots, one digit bit at a time; LDS
//                       counters per wave keep the order), puts them in digit order in LDS and
//                       writes runs of equal digits to their places
// Bound: the entries' bytes, read and written once a pass, and at these sizes the launches.
// Measured there: 57 us for the 1.65M float64 entries (histograms 11, scans 8, scatters 37, 2.8
// TB/s of what they read and write) and 47 us for the 1.2M float32 ones; the whole SpMV call 1551
// -> 111 us, the SpMM call of N = 32 452 -> 111 us.
#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

constexpr int kSortBlock = 512;
constexpr int kSortWaves = kSortBlock / kWave;
// Entries per thread of a tile: 4 for short sorts, whose tiles would not fill the CUs, else 8 (runs
// of equal digits twice as long).  Measured on MI355X, a sort with 4 / 8: 16k entries 20.2 / 24.5
// us, 400k 26.4 / 33.7, 1.65M 56.4 / 52.4, 12M 336 / 285.
constexpr int kShortSteps = 4, kLongSteps = 8;
constexpr int64_t kShortNnz = 1 << 20;
constexpr int kMaxDigits = 512;  // one per thread in the scatter kernel's scans
static_assert(kMaxDigits == kSortBlock, "a thread per digit");
// Up to this many tiles the scatter kernel reads all their counts itself: a launch less, which a
// small sort is made of (two passes of 16k entries: 29.4 -> 20.8 us of host time with the launches).
constexpr int kFewTiles = 32;

__device__ __forceinline__ int wave_inclusive(int v) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(v, off, kWave);
    if (lane >= off) v += o;
  }
  return v;
}

// Exclusive sum of v over the workgroup's threads in thread order, and the total; s_w holds an
// int per wave.
template <int WAVES>
__device__ __forceinline__ int block_exclusive(int v, int* s_w, int* total) {
  const int incl = wave_inclusive(v);
  const int w = threadIdx.x / kWave;
  __syncthreads();  // s_w may still be read by a previous call
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_w[w] = incl;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    before += i < w ? s_w[i] : 0;
    all += s_w[i];
  }
  *total = all;
  return before + incl - v;
}

template <typename R, int STEPS>
__global__ __launch_bounds__(kSortBlock) void coo_hist_kernel(const R* __restrict__ rows, int n,
                                                              int shift, int bits, int n_tiles,
                                                              int* __restrict__ counts) {
  constexpr int TILE = kSortBlock * STEPS;
  __shared__ int s_cnt[kMaxDigits];
  const int tile = xcd_logical_block(blockIdx.x, n_tiles);  // neighbours share lines of counts
  const int D = 1 << bits;
  if ((int)threadIdx.x < D) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  const int base = tile * TILE;
  int d[STEPS];
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    const int i = base + q * kSortBlock + threadIdx.x;  // < 2^31: n <= 2^31 - 1 - TILE
    d[q] = i < n ? (int)((uint32_t)rows[i] >> shift) & (D - 1) : -1;
  }
#pragma unroll
  for (int q = 0; q < STEPS; ++q)
    if (d[q] >= 0) atomicAdd(&s_cnt[d[q]], 1);
  __syncthreads();
  if ((int)threadIdx.x < D) counts[(int64_t)threadIdx.x * n_tiles + tile] = s_cnt[threadIdx.x];
}

__global__ __launch_bounds__(kBlock) void coo_scan_kernel(int* __restrict__ counts, int n_tiles,
                                                          int* __restrict__ totals) {
  __shared__ int s_w[kWavesPerBlock];
  int* c = counts + (int64_t)blockIdx.x * n_tiles;
  int run = 0;
  for (int t0 = 0; t0 < n_tiles; t0 += kBlock) {
    const int t = t0 + threadIdx.x;
    int total;
    const int ex = block_exclusive<kWavesPerBlock>(t < n_tiles ? c[t] : 0, s_w, &total);
    if (t < n_tiles) c[t] = run + ex;
    run += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

template <typename R, typename C, typename T, int STEPS>
__global__ __launch_bounds__(kSortBlock) void coo_scatter_kernel(
    const R* __restrict__ rows, const C* __restrict__ cols, const T* __restrict__ vals, int n,
    int shift, int bits, int n_tiles, const int* __restrict__ counts,
    const int* __restrict__ totals, int* __restrict__ out_rows, int* __restrict__ out_cols,
    T* __restrict__ out_vals) {
  constexpr int TILE = kSortBlock * STEPS;
  __shared__ int s_key[TILE];
  __shared__ T s_buf[TILE];  // the columns, then the values, in digit order
  __shared__ uint16_t s_cnt[kSortWaves][kMaxDigits];
  __shared__ int s_start[kMaxDigits];  // a digit's first position in the tile's digit order
  __shared__ int s_dst[kMaxDigits];    // its place in the output, less s_start
  __shared__ int s_w[kSortWaves];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  const int tile = xcd_logical_block(blockIdx.x, n_tiles);
  const int D = 1 << bits, base = tile * TILE;
  const int m = n - base < TILE ? n - base : TILE;
  int key[STEPS], col[STEPS];
  T val[STEPS];
  int at[STEPS];  // wave w holds entries [w * 512, w * 512 + 512) in order, 64 a step
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    const int i = w * (TILE / kSortWaves) + q * kWave + lane;
    const bool ok = i < m;
    key[q] = ok ? (int)rows[base + i] : 0;
    col[q] = ok ? (int)cols[base + i] : 0;
    val[q] = ok ? vals[base + i] : T(0);
  }
  for (int i = tid; i < kSortWaves * kMaxDigits; i += kSortBlock)
    (&s_cnt[0][0])[i] = 0;
  __syncthreads();
  volatile uint16_t* cnt = s_cnt[w];
  const uint64_t below = (uint64_t(1) << lane) - 1;
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    const bool ok = w * (TILE / kSortWaves) + q * kWave + lane < m;
    const int d = (int)((uint32_t)key[q] >> shift) & (D - 1);
    uint64_t same = __ballot(ok);  // the lanes of this step that hold the same digit
    for (int b = 0; b < bits; ++b) {
      const bool bit = (d >> b) & 1;
      const uint64_t vote = __ballot(bit);
      same &= bit ? vote : ~vote;
    }
    int have = 0;
    if (ok) have = cnt[d];
    at[q] = have + __popcll(same & below);
    __builtin_amdgcn_wave_barrier();
    if (ok && (same & below) == 0) cnt[d] = (uint16_t)(have + __popcll(same));
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // Thread d: digit d's counts of the waves become the waves' offsets; the tile's digit starts
  // and the digits' places in the output are exclusive sums over the digits.
  int mine = 0;
  if (tid < D) {
#pragma unroll
    for (int v = 0; v < kSortWaves; ++v) {
      const int c = s_cnt[v][tid];
      s_cnt[v][tid] = (uint16_t)mine;
      mine += c;
    }
  }
  // The digit's entries in all tiles and in those before this one: from coo_scan_kernel, or,
  // where tiles are few (totals NULL), added up here.
  int in_all = 0, in_before = 0;
  if (tid < D) {
    if (totals) {
      in_all = totals[tid];
      in_before = counts[(int64_t)tid * n_tiles + tile];
    } else {
      for (int t = 0; t < n_tiles; ++t) {
        const int c = counts[(int64_t)tid * n_tiles + t];
        in_all += c;
        in_before += t < tile ? c : 0;
      }
    }
  }
  int all;
  const int start = block_exclusive<kSortWaves>(mine, s_w, &all);
  const int place = block_exclusive<kSortWaves>(in_all, s_w, &all);
  if (tid < D) {
    s_start[tid] = start;
    s_dst[tid] = place + in_before - start;
  }
  __syncthreads();
  int* s_col = reinterpret_cast<int*>(s_buf);
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    if (w * (TILE / kSortWaves) + q * kWave + lane < m) {
      const int d = (int)((uint32_t)key[q] >> shift) & (D - 1);
      at[q] += s_start[d] + s_cnt[w][d];
      s_key[at[q]] = key[q];
      s_col[at[q]] = col[q];
    }
  }
  __syncthreads();
  int dst[STEPS];
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    const int i = q * kSortBlock + tid;
    dst[q] = -1;
    if (i < m) {
      const int k = s_key[i];
      dst[q] = s_dst[(int)((uint32_t)k >> shift) & (D - 1)] + i;
      out_rows[dst[q]] = k;
      out_cols[dst[q]] = s_col[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < STEPS; ++q)
    if (w * (TILE / kSortWaves) + q * kWave + lane < m) s_buf[at[q]] = val[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < STEPS; ++q)
    if (dst[q] >= 0) out_vals[dst[q]] = s_buf[q * kSortBlock + tid];
}

// The number of entries in rows[lo, hi) whose row is below r, plus lo, by one wave: 64 probes at a
// time, so a search of n entries is log65(n) loads deep instead of log2(n).
template <typename R>
__device__ inline int64_t wave_lower_bound(const R* __restrict__ rows, int64_t lo, int64_t hi,
                                           int64_t r, int lane) {
  while (lo < hi) {
    const int64_t step = (hi - lo + 64) / 65;
    const int64_t probe = lo + (lane + 1) * step - 1;
    const bool below = probe < hi && (int64_t)rows[probe] < r;
    const int64_t c = __popcll(__ballot(below));
    const int64_t end = lo + (c + 1) * step - 1;
    lo += c * step;
    if (c < 64 && end < hi) hi = end;  // rows[end] >= r; after 64 probes nothing is known of hi
  }
  return lo;
}

template <typename R>
__device__ inline int64_t lower_bound(const R* __restrict__ rows, int64_t lo, int64_t hi, int64_t r) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)rows[mid] < r) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// ptr[r] = the number of entries whose row is below r: one binary search per row.
template <typename R, typename P>
__global__ __launch_bounds__(kBlock) void coo_rowptr_search_kernel(const R* __restrict__ rows,
                                                                   int64_t n, int64_t n_rows,
                                                                   P* __restrict__ ptr) {
  const int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (r <= n_rows) ptr[r] = (P)lower_bound(rows, (int64_t)0, n, r);
}

// The same pointers from one read of the entries.  A workgroup takes 256 pointers: two waves search
// for the first and the last, then the entries between them are read in order, four to a lane, and
// each place where the row rises writes the pointers up to the new row.  More than kRowptrScan
// entries between them (a long row, or rows far above the average) are searched by a thread per
// pointer instead, so no workgroup reads a long row alone.
// MI355X, int32, us, a search per row -> this kernel:
//   33.5M entries in 1M rows     62.7 -> 34.8  (one read at the copy's rate: 27)
//   the same, power-law lengths  36.0 -> 24.0
//   2M entries in 2M rows        20.1 -> 17.0
//   1.2M entries in 150,000 rows  6.0 -> 5.4
// It is not used where it was slower: below kRowptrScanRows rows a search per row finds its first
// steps in L2 and the launch is all latency (600,000 entries in 60,000 rows 4.3 against 4.5, 16.8M
// in 1000 rows 5.3 against 6.3), and with more rows than entries the runs of empty rows are
// written by the one lane that meets them (400,000 entries in 4M rows 31.6 against 46.6).
constexpr int64_t kRowptrScan = 64 * kBlock;
constexpr int64_t kRowptrScanRows = int64_t(1) << 17;

template <typename R, typename P>
__global__ __launch_bounds__(kBlock) void coo_rowptr_kernel(const R* __restrict__ rows, int64_t n,
                                                            int64_t n_rows, P* __restrict__ ptr) {
  __shared__ int64_t s_ends[2];
  __shared__ int s_at[kBlock];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * kBlock;
  const int64_t last = r0 + kBlock - 1 < n_rows ? r0 + kBlock - 1 : n_rows;
  if (wave < 2) {
    const int64_t e = wave_lower_bound(rows, (int64_t)0, n, wave == 0 ? r0 : last, lane);
    if (lane == 0) s_ends[wave] = e;
  }
  __syncthreads();
  const int64_t lo = s_ends[0], hi = s_ends[1];
  const int64_t r = r0 + tid;
  if (hi - lo > kRowptrScan) {
    if (r > n_rows) return;
    ptr[r] = (P)lower_bound(rows, lo, hi, r);
    return;
  }
  s_at[tid] = tid == 0 ? 0 : (int)(hi - lo);
  __syncthreads();
  // every entry here lies in a row of [r0, last), so the pointers written are those of (r0, last)
  for (int64_t p = lo + 4 * tid; p < hi; p += 4 * kBlock) {
    R row[4];
    if (p + 4 <= hi) {
#pragma unroll
      for (int j = 0; j < 4; ++j) row[j] = rows[p + j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) row[j] = rows[p + j < hi ? p + j : hi - 1];
    }
    R before = p > lo ? rows[p - 1] : (R)r0;
    if (before == row[3]) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // for rows in order r0 <= before <= row < r0 + kBlock; held to that, no write leaves s_at
      const int from = before < (R)r0 ? 0 : before < (R)last ? (int)(before - (R)r0) : kBlock - 1;
      const int to = row[j] < (R)r0 ? 0 : row[j] < (R)last ? (int)(row[j] - (R)r0) : kBlock - 1;
      for (int k = from + 1; k <= to; ++k) s_at[k] = (int)(p + j - lo);
      before = row[j];
    }
  }
  __syncthreads();
  if (r <= n_rows) ptr[r] = (P)(lo + s_at[tid]);
}

template <typename R, typename P>
int launch_rowptr(const void* rows, int64_t nnz, int64_t n_rows, void* ptr, hipStream_t st) {
  const dim3 grid((unsigned)(n_rows / kBlock + 1)), block(kBlock);
  const R* r = static_cast<const R*>(rows);
  P* p = static_cast<P*>(ptr);
  if (n_rows >= kRowptrScanRows && nnz >= n_rows)
    hipLaunchKernelGGL((coo_rowptr_kernel<R, P>), grid, block, 0, st, r, nnz, n_rows, p);
  else
    hipLaunchKernelGGL((coo_rowptr_search_kernel<R, P>), grid, block, 0, st, r, nnz, n_rows, p);
  return check_hip(hipGetLastError(), "coo_rowptr_kernel launch");
}

struct SortPlan {
  int passes, bits, steps, n_tiles;  // bits per pass, entries per thread
};

SortPlan sort_plan(int64_t nnz, int64_t max_row) {
  int bits = 1;
  while (bits < 31 && (max_row >> bits) != 0) ++bits;
  SortPlan p;
  p.passes = (bits + 8) / 9;
  p.bits = (bits + p.passes - 1) / p.passes;
  p.steps = nnz < kShortNnz ? kShortSteps : kLongSteps;
  const int64_t tile = (int64_t)kSortBlock * p.steps;
  p.n_tiles = (int)((nnz + tile - 1) / tile);
  return p;
}

int64_t align16(int64_t b) { return (b + 15) & ~int64_t(15); }

template <typename R, typename C, typename T, int STEPS>
int sort_pass_steps(const R* rows, const C* cols, const T* vals, int n, int shift, const SortPlan& p,
              int* counts, int* totals, int* out_rows, int* out_cols, T* out_vals,
              hipStream_t st) {
  const unsigned tiles = (unsigned)p.n_tiles;
  hipLaunchKernelGGL((coo_hist_kernel<R, STEPS>), dim3(tiles), dim3(kSortBlock), 0, st, rows, n, shift,
                     p.bits, p.n_tiles, counts);
  int rc = check_hip(hipGetLastError(), "coo_hist_kernel launch");
  if (rc) return rc;
  if (p.n_tiles <= kFewTiles) {
    totals = nullptr;  // the scatter kernel adds the counts up
  } else {
    hipLaunchKernelGGL(coo_scan_kernel, dim3(1u << p.bits), dim3(kBlock), 0, st, counts,
                       p.n_tiles, totals);
    rc = check_hip(hipGetLastError(), "coo_scan_kernel launch");
    if (rc) return rc;
  }
  hipLaunchKernelGGL((coo_scatter_kernel<R, C, T, STEPS>), dim3(tiles), dim3(kSortBlock), 0, st, rows,
                     cols, vals, n, shift, p.bits, p.n_tiles, counts, totals, out_rows, out_cols,
                     out_vals);
  return check_hip(hipGetLastError(), "coo_scatter_kernel launch");
}

template <typename R, typename C, typename T>
int sort_pass(const R* rows, const C* cols, const T* vals, int n, int shift, const SortPlan& p,
              int* counts, int* totals, int* out_rows, int* out_cols, T* out_vals,
              hipStream_t st) {
  if (p.steps == kShortSteps)
    return sort_pass_steps<R, C, T, kShortSteps>(rows, cols, vals, n, shift, p, counts, totals,
                                                 out_rows, out_cols, out_vals, st);
  return sort_pass_steps<R, C, T, kLongSteps>(rows, cols, vals, n, shift, p, counts, totals,
                                              out_rows, out_cols, out_vals, st);
}

template <typename R, typename C, typename T>
int sort_rows(const void* rows, const void* cols, const void* vals, int64_t nnz, int64_t max_row,
              int32_t* out_rows, int32_t* out_cols, void* out_vals, void* scratch,
              hipStream_t st) {
  const SortPlan p = sort_plan(nnz, max_row);
  const int n = (int)nnz;
  char* s = static_cast<char*>(scratch);
  T* tmp_vals = reinterpret_cast<T*>(s);
  s += align16(nnz * (int64_t)sizeof(T));
  int* tmp_rows = reinterpret_cast<int*>(s);
  s += align16(nnz * 4);
  int* tmp_cols = reinterpret_cast<int*>(s);
  s += align16(nnz * 4);
  int* totals = reinterpret_cast<int*>(s);
  int* counts = totals + kMaxDigits;
  // the passes alternate between the outputs and the scratch copies and end in the outputs
  bool to_out = p.passes % 2 == 1;
  for (int i = 0; i < p.passes; ++i, to_out = !to_out) {
    int* r = to_out ? out_rows : tmp_rows;
    int* c = to_out ? out_cols : tmp_cols;
    T* v = to_out ? static_cast<T*>(out_vals) : tmp_vals;
    const int* fr = to_out ? tmp_rows : out_rows;
    const int* fc = to_out ? tmp_cols : out_cols;
    const T* fv = to_out ? tmp_vals : static_cast<const T*>(out_vals);
    const int rc = i == 0
                       ? sort_pass<R, C, T>(static_cast<const R*>(rows), static_cast<const C*>(cols),
                                            static_cast<const T*>(vals), n, 0, p, counts, totals, r,
                                            c, v, st)
                       : sort_pass<int32_t, int32_t, T>(fr, fc, fv, n, i * p.bits, p, counts,
                                                        totals, r, c, v, st);
    if (rc) return rc;
  }
  return FSP_OK;
}

template <typename T>
int sort_any(int row_bits, int col_bits, const void* rows, const void* cols, const void* vals,
             int64_t nnz, int64_t max_row, int32_t* out_rows, int32_t* out_cols, void* out_vals,
             void* scratch, hipStream_t st) {
#define FSP_SORT(RR, CC) \
  return sort_rows<RR, CC, T>(rows, cols, vals, nnz, max_row, out_rows, out_cols, out_vals, scratch, st)
  if (row_bits == 32 && col_bits == 32) FSP_SORT(int32_t, int32_t);
  if (row_bits == 32) FSP_SORT(int32_t, int64_t);
  if (col_bits == 32) FSP_SORT(int64_t, int32_t);
  FSP_SORT(int64_t, int64_t);
#undef FSP_SORT
}

}  // namespace
}  // namespace fsp

using namespace fsp;

extern "C" int64_t fsp_coo_sort_max_nnz(void) { return 0x7fffffffLL - kSortBlock * kLongSteps; }

extern "C" int64_t fsp_coo_sort_scratch(int dtype, int64_t nnz, int64_t max_row) {
  if (nnz < 1 || nnz > fsp_coo_sort_max_nnz() || max_row < 0) return 0;
  const SortPlan p = sort_plan(nnz, max_row);
  return align16(nnz * (dtype == FSP_F64 ? 8 : 4)) + 2 * align16(nnz * 4) +
         4 * (kMaxDigits + ((int64_t)p.n_tiles << p.bits));
}

extern "C" int fsp_coo_sort_rows(int dtype, const void* rows, int row_bits, const void* cols,
                                 int col_bits, const void* vals, int64_t nnz, int64_t max_row,
                                 int32_t* out_rows, int32_t* out_cols, void* out_vals,
                                 void* scratch, void* stream) {
  if (dtype != FSP_F32 && dtype != FSP_F64)
    return set_error(FSP_ENOTSUP, "fsp_coo_sort_rows: dtype");
  if ((row_bits != 32 && row_bits != 64) || (col_bits != 32 && col_bits != 64))
    return set_error(FSP_EINVAL, "fsp_coo_sort_rows: index widths must be 32 or 64");
  if (nnz < 0 || nnz > fsp_coo_sort_max_nnz() || max_row < 0 || max_row > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_coo_sort_rows: size out of range");
  if (nnz == 0) return FSP_OK;
  if (!rows || !cols || !vals || !out_rows || !out_cols || !out_vals || !scratch)
    return set_error(FSP_EINVAL, "fsp_coo_sort_rows: null pointer");
  if (reinterpret_cast<uintptr_t>(scratch) % 16)
    return set_error(FSP_EINVAL, "fsp_coo_sort_rows: scratch must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == FSP_F32)
    return sort_any<float>(row_bits, col_bits, rows, cols, vals, nnz, max_row, out_rows, out_cols,
                           out_vals, scratch, st);
  return sort_any<double>(row_bits, col_bits, rows, cols, vals, nnz, max_row, out_rows, out_cols,
                          out_vals, scratch, st);
}

extern "C" int fsp_coo_rowptr(const void* rows, int row_bits, int64_t nnz, int64_t n_rows,
                              void* ptr, int ptr_bits, void* stream) {
  if ((row_bits != 32 && row_bits != 64) || (ptr_bits != 32 && ptr_bits != 64))
    return set_error(FSP_EINVAL, "fsp_coo_rowptr: index widths must be 32 or 64");
  if (nnz < 0 || n_rows < 0 || n_rows > 0x7fffffffLL || (ptr_bits == 32 && nnz > 0x7fffffffLL))
    return set_error(FSP_EINVAL, "fsp_coo_rowptr: size out of range");
  if (!ptr || (nnz > 0 && !rows)) return set_error(FSP_EINVAL, "fsp_coo_rowptr: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (row_bits == 32 && ptr_bits == 32)
    return launch_rowptr<int32_t, int32_t>(rows, nnz, n_rows, ptr, st);
  if (row_bits == 32) return launch_rowptr<int32_t, int64_t>(rows, nnz, n_rows, ptr, st);
  if (ptr_bits == 32) return launch_rowptr<int64_t, int32_t>(rows, nnz, n_rows, ptr, st);
  return launch_rowptr<int64_t, int64_t>(rows, nnz, n_rows, ptr, st);
}
