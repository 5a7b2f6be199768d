// CSR SpMV without a plan: the matrix cut into slices of about equal work, for calls that use
// a matrix once (no prepared object) and for prepared matrices with very uneven rows.
//
// Reference behaviour followed (src/flagsparse/sparse_operations/):
//   spmv_csr.py:94-120    y[row] = sum over the row's entries, float32 summed in float64
//   spmv_csr.py:161-279   use_opt: summed in the input type
//   spmv_coo.py:51-108    one output row per run of equal rows, rows without entries 0
//
// A row-block plan costs two passes over the row pointers, prefix sums and a host wait for the
// table sizes.  Here the number of slices is known from the sizes alone: the rows and entries
// are laid on one line in which row r takes the positions rowptr[r] + r .. rowptr[r+1] + r (its
// entries, then its end), and slice k starts at position k * W.  slice_table_kernel finds the
// row there by binary search.  (The line is that of merge-based CSR SpMV, Merrill and Garland,
// SC 2016; here whole rows are kept together where they can be.)  A boundary inside a row of at
// most T entries moves to that row's start, so only longer rows are cut; a slice holds at most
// W + T + 3 rows and entries together, whatever the row lengths, empty rows included.
//
// spmv_slices_kernel: a workgroup reads its slice's entries with 16-byte loads, leaves the
// products in LDS and sums its rows (G lanes each, rows much longer than their neighbours a
// wave each, in a second step).  The piece of a row that continues in the next slice goes to
// carry[k]; the end of a row that began in an earlier slice to head[k]; slice_fixup_kernel adds
// the pieces of such rows in slice order (deterministic).
//
// Bound: the entries' stream and the x gathers, as spmv_rowblock_kernel.  Measured on MI355X, a
// power law of 1.0M rows and 12.0M entries (float32 summed in float64, x of 4 MB, int64
// indices): the whole call 1049 -> 130 us; of it the table 8, the product 62.5 (row blocks: 90.5,
// whose many short rows and few long ones share a block badly), the second pass 5.1.
#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

constexpr int kSlots = (int)kSpmvSliceSlots;
constexpr int kUPT = kSlots / (4 * kBlock);  // quads of entries per thread
static_assert(kUPT * 4 * kBlock == kSlots, "slice slots must be whole quads per thread");
static_assert(kSpmvSliceItems + kSpmvSliceKeep + 3 <= kSlots - 3, "a slice must fit the slots");
constexpr int kPtrPT = (kSlots + kBlock) / kBlock;  // row pointers per thread

// One boundary per 8 lanes, which probe 8 rows at a time: 7 dependent reads for a million rows
// where bisection has 20 (17k boundaries of a 1M-row matrix on MI355X: 8.1 us by bisection, 4.6
// us so; every level but the last two is in the cache).
constexpr int kProbe = 8;

template <typename P>
__global__ __launch_bounds__(kBlock) void slice_table_kernel(const P* __restrict__ rowptr,
                                                             int64_t n_rows, int64_t nnz,
                                                             int64_t W, int64_t T,
                                                             int64_t n_slices,
                                                             int64_t* __restrict__ table) {
  const int lane = threadIdx.x & (kWave - 1), mine = lane & (kProbe - 1);
  const int64_t k = (int64_t)blockIdx.x * (kBlock / kProbe) + threadIdx.x / kProbe;
  if (k > n_slices) return;  // the same for a boundary's 8 lanes
  int64_t row = n_rows, pos = nnz;
  if (k < n_slices) {
    const int64_t d = k * W;  // < n_rows + nnz
    int64_t lo = 0, hi = n_rows;  // the largest i with rowptr[i] + i <= d (true for i = 0)
    while (lo < hi) {
      const int64_t step = (hi - lo + kProbe - 1) / kProbe;
      const int64_t at = lo + (mine + 1) * step < hi ? lo + (mine + 1) * step : hi;
      const uint64_t vote = __ballot((int64_t)rowptr[at] + at <= d);
      const int c = __popcll((vote >> (lane - mine)) & ((1u << kProbe) - 1));
      const int64_t next = lo + (c + 1) * step - 1;
      lo = lo + c * step < hi ? lo + c * step : hi;
      hi = c < kProbe && next < hi ? next : hi;
    }
    row = lo;
    if (row < n_rows) {
      const int64_t a = (int64_t)rowptr[row], e = (int64_t)rowptr[row + 1];
      pos = a;
      if (e - a > T) {  // a long row is cut, at a multiple of 4 entries
        const int64_t j = (d - row) & ~int64_t(3);
        pos = j > a ? j : a;
      }
    }
  }
  if (mine == 0) {
    table[2 * k] = row;
    table[2 * k + 1] = pos;
  }
}

// Launch order of the slices for products whose dense operand does not fit an L2.  A slice that
// lies inside one long row reads a narrow range of columns (CSR rows in column order: 512 of
// 50,000 entries cover 1 % of them), and the long rows of a power law all read the same ranges.
// In row order no two of them meet in an L2 before the lines are gone.  The order puts the other
// slices first, in row order, then those inside one row by the column they start at; each XCD
// (launch slot b runs on XCD b mod 8) takes one contiguous eighth of either part, so an XCD reads
// one eighth of the dense operand for the long rows, a moving window of it at a time.  It changes
// only when a slice runs, never a sum.  Unordered columns make a poor order, nothing worse.
// Measured on MI355X, row order / this order: SpMM of a power law, fp32 N=47, 4.8M entries (B of
// 38 MB) 214 / 125 us, N=128, 3.6M 332 / 190; SDDMM fp32 K=128, 4.8M 352 / 189.  The long slices
// first: 130 and 202 us.  Three launches, a counting sort on 256 column bins: 14 us for 8k.
constexpr int kBins = 256;  // bin 0: not inside one row

// Slices per workgroup of the counting sort: few for short launches (8k slices with 1024: 17 us
// for the three launches instead of 14), more where the counts would make the scan long.
int64_t order_tile(int64_t n) { return n <= (1 << 14) ? kBlock : 4 * kBlock; }

__device__ __forceinline__ int column_bin(int col, int64_t n_cols) {
  const int64_t b = (int64_t)col * (kBins - 1) / n_cols;
  return 1 + (int)(b < 0 ? 0 : b > kBins - 2 ? kBins - 2 : b);
}

// What is ordered: slices (the order is of their numbers) ...
struct Slices {
  const int64_t* table;
  const int* cols;
  int64_t n_cols;
  int* order;
  __device__ __forceinline__ int bin(int64_t k) const {
    const int64_t i0 = table[2 * k], p0 = table[2 * k + 1];
    if (table[2 * k + 2] != i0 || table[2 * k + 3] <= p0) return 0;
    return column_bin(cols[p0], n_cols);
  }
  __device__ __forceinline__ void put(int64_t slot, int64_t k) const { order[slot] = (int)k; }
};

// ... or a row-block plan's descriptors {first row, .., 0, ..} and {long row, part, parts, ..},
// of which the parts go by column (moved themselves: out must be another array).
template <typename P>
struct Descriptors {
  const i32x4* desc;
  const P* rowptr;
  int64_t chunk;
  const int* cols;
  int64_t n_cols;
  i32x4* out;
  __device__ __forceinline__ int bin(int64_t k) const {
    const i32x4 d = desc[k];
    if (d.z <= 0) return 0;
    return column_bin(cols[(int64_t)rowptr[d.x] + d.y * chunk], n_cols);
  }
  __device__ __forceinline__ void put(int64_t slot, int64_t k) const { out[slot] = desc[k]; }
};

template <typename S>
__global__ __launch_bounds__(kBlock) void order_hist_kernel(S what, int64_t n, int tile,
                                                            int n_tiles,
                                                            int* __restrict__ counts) {
  __shared__ int s_cnt[kBins];
  s_cnt[threadIdx.x] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < tile; i += kBlock) {
    const int64_t k = (int64_t)blockIdx.x * tile + i;
    if (k < n) atomicAdd(&s_cnt[what.bin(k)], 1);
  }
  __syncthreads();
  counts[(int64_t)threadIdx.x * n_tiles + blockIdx.x] = s_cnt[threadIdx.x];
}

// Exclusive sums over all (bin, tile) counts, bins outer (or over the slices' pieces): one
// workgroup.
__global__ __launch_bounds__(1024) void order_scan_kernel(int* __restrict__ counts, int64_t m) {
  __shared__ int s_w[1024 / kWave];
  int run = 0;
  for (int64_t b = 0; b < m; b += 4096) {
    int v[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t i = b + 4 * threadIdx.x + j;
      v[j] = i < m ? counts[i] : 0;
      sum += v[j];
    }
    int incl = sum;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int o = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += o;
    }
    __syncthreads();  // the previous step's reads of s_w
    if (lane == kWave - 1) s_w[w] = incl;
    __syncthreads();
    int before = run, all = 0;
#pragma unroll
    for (int i = 0; i < 1024 / kWave; ++i) {
      before += i < w ? s_w[i] : 0;
      all += s_w[i];
    }
    before += incl - sum;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t i = b + 4 * threadIdx.x + j;
      if (i < m) counts[i] = before;
      before += v[j];
    }
    run += all;
  }
}

// Position p of q slices cut into eight contiguous parts, part x on XCD x: its launch slot (the
// inverse of xcd_logical_block).
__device__ __forceinline__ int64_t xcd_slot(int64_t p, int64_t q) {
  const int64_t per = q / 8, r = q % 8, big = r * (per + 1);
  const int64_t x = p < big ? p / (per + 1) : r + (p - big) / per;
  const int64_t j = p < big ? p % (per + 1) : (p - big) % per;
  return 8 * j + x;
}

template <typename S>
__global__ __launch_bounds__(kBlock) void order_scatter_kernel(S what, int64_t n, int tile,
                                                               int n_tiles,
                                                               const int* __restrict__ places) {
  __shared__ int s_cnt[kBins];
  s_cnt[threadIdx.x] = places[(int64_t)threadIdx.x * n_tiles + blockIdx.x];
  __syncthreads();
  const int64_t others = places[n_tiles];  // bin 1 starts there: the slices of bin 0
  for (int i = threadIdx.x; i < tile; i += kBlock) {
    const int64_t k = (int64_t)blockIdx.x * tile + i;
    if (k < n) {
      const int64_t p = atomicAdd(&s_cnt[what.bin(k)], 1);
      const int64_t slot = p < others ? xcd_slot(p, others)
                                      : others + xcd_slot(p - others, n - others);
      what.put(slot, k);
    }
  }
}

template <typename S>
int launch_order(const S& what, int64_t n, int32_t* scratch, hipStream_t st) {
  const int tile = (int)order_tile(n);
  const int tiles = (int)((n + tile - 1) / tile);
  hipLaunchKernelGGL((order_hist_kernel<S>), dim3((unsigned)tiles), dim3(kBlock), 0, st, what, n,
                     tile, tiles, scratch);
  int rc = check_hip(hipGetLastError(), "order_hist_kernel launch");
  if (rc) return rc;
  hipLaunchKernelGGL(order_scan_kernel, dim3(1), dim3(1024), 0, st, scratch,
                     (int64_t)kBins * tiles);
  rc = check_hip(hipGetLastError(), "order_scan_kernel launch");
  if (rc) return rc;
  hipLaunchKernelGGL((order_scatter_kernel<S>), dim3((unsigned)tiles), dim3(kBlock), 0, st, what,
                     n, tile, tiles, scratch);
  return check_hip(hipGetLastError(), "order_scatter_kernel launch");
}

// The pieces of cut rows that slice k holds: the end of a row begun earlier, the start of a row that
// goes on in the next slice.  What spmm_slices_kernel puts into head[k] and carry[k].
template <typename P>
__global__ __launch_bounds__(kBlock) void slice_piece_count_kernel(
    const P* __restrict__ rowptr, const int64_t* __restrict__ table, int64_t n,
    int* __restrict__ counts) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k > n) return;
  int c = 0;
  if (k < n) {
    const int64_t i0 = table[2 * k], p0 = table[2 * k + 1];
    const int64_t i1 = table[2 * k + 2], p1 = table[2 * k + 3];
    if (i1 > i0 && (int64_t)rowptr[i0] < p0) ++c;
    const int64_t a = (int64_t)rowptr[i1];
    if (p1 > (a > p0 ? a : p0)) ++c;
  }
  counts[k] = c;
}

template <typename T, typename A, typename P>
__global__ __launch_bounds__(kBlock) void spmv_slices_kernel(
    const T* __restrict__ vals, const int* __restrict__ cols, const P* __restrict__ rowptr,
    P nnz_total, const T* __restrict__ x, T* __restrict__ y, const int64_t* __restrict__ table,
    A* __restrict__ carry, A* __restrict__ head) {
  __shared__ A s_prod[kSlots];
  __shared__ int s_ptr[kSlots + 2];
  // Rows left for the second step: longer than 16 G entries each, so at most kSlots / 16.
  __shared__ int s_list[kSlots / 16];
  __shared__ int s_n;
  const int tid = threadIdx.x;
  const int64_t k = blockIdx.x;
  const int64_t i0 = table[2 * k], i1 = table[2 * k + 2];
  const P p0 = (P)table[2 * k + 1], p1 = (P)table[2 * k + 3];
  const int64_t R64 = i1 - i0;
  if (R64 < 0 || R64 > kSlots || p1 < p0 || p1 - p0 > P(kSlots - 3)) return;  // uniform
  const int R = (int)R64, n = (int)(p1 - p0);
  const P s0 = p0 & ~P(3);

  T v[kUPT][4];
  int c[kUPT][4];
#pragma unroll
  for (int u = 0; u < kUPT; ++u) {
    const Wide<P> base = Wide<P>(s0) + 4 * (tid + u * kBlock);
    if (base < Wide<P>(p1)) {
      QuadLoader<false, T>::load(vals, cols, P(base), p0, p1, nnz_total, v[u], c[u]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) { v[u][j] = T(0); c[u][j] = -1; }
    }
  }
  // The slice's row starts, relative to p0: position s of rows i0 + s, s = 0 .. R.
  int rp[kPtrPT];
#pragma unroll
  for (int u = 0; u < kPtrPT; ++u) {
    const int s = tid + u * kBlock;
    rp[u] = 0;
    if (s <= R) {
      const P a = rowptr[i0 + s];
      rp[u] = a > p0 ? (int)(a - p0) : 0;
    }
  }
  const bool begun = R > 0 && rowptr[i0] < p0;  // row i0 began in an earlier slice and ends here
  T xv[kUPT][4];
  gather_x<kUPT, A>(x, c, n > 0, xv);
#pragma unroll
  for (int u = 0; u < kUPT; ++u) {
    const Wide<P> base = Wide<P>(s0) + 4 * (tid + u * kBlock);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (c[u][j] >= 0) s_prod[(int)(base + j - Wide<P>(p0))] = A(v[u][j]) * A(xv[u][j]);
  }
#pragma unroll
  for (int u = 0; u < kPtrPT; ++u) {
    const int s = tid + u * kBlock;
    if (s <= R) s_ptr[s] = rp[u];
  }
  if (tid == 0) {
    s_ptr[R + 1] = n;
    s_n = 0;
  }
  __syncthreads();

  // R finished rows and the piece of row i1 that this slice holds (often empty): G lanes each,
  // G the largest power of two <= 64 with G * next_pow2(R + 1) <= 256.
  int lg = 0;
  if (R + 1 < kBlock) {
    int p2 = 1, lp = 0;
    while (p2 < R + 1) { p2 <<= 1; ++lp; }
    lg = 8 - lp;
    if (lg > 6) lg = 6;
  }
  const int G = 1 << lg, ngrp = kBlock >> lg;
  const int grp = tid >> lg, lane = tid & (G - 1);
  auto put = [&](int s, A sum) {
    if (s == R) carry[k] = sum;
    else if (s == 0 && begun) head[k] = sum;
    else y[i0 + s] = T(sum);
  };
  for (int s = grp; s <= R; s += ngrp) {
    const int a = s_ptr[s], e = s_ptr[s + 1];
    if (lg < 6 && e - a > 16 * G) {
      if (lane == 0) s_list[atomicAdd(&s_n, 1)] = s;
    } else {
      A acc = A(0);
      for (int i = a + lane; i < e; i += G) acc += s_prod[i];
      if (G > 1) acc = group_sum(acc, G);
      if (lane == 0) put(s, acc);
    }
  }
  __syncthreads();
  const int n_long = s_n;
  for (int l = tid / kWave; l < n_long; l += kWavesPerBlock) {
    const int s = s_list[l];
    const int a = s_ptr[s], e = s_ptr[s + 1];
    A acc = A(0);
    for (int i = a + (tid & (kWave - 1)); i < e; i += kWave) acc += s_prod[i];
    acc = wave_sum(acc);
    if ((tid & (kWave - 1)) == 0) put(s, acc);
  }
}

// A wave per slice: when the slice ends a row that began in an earlier one, y[row] = the
// carries of the slices the row began in and crossed, in a fixed order, plus this head.
template <typename T, typename A, typename P>
__global__ __launch_bounds__(kBlock) void spmv_slice_fixup_kernel(
    const P* __restrict__ rowptr, const int64_t* __restrict__ table, int64_t n_slices, int64_t W,
    const A* __restrict__ carry, const A* __restrict__ head, T* __restrict__ y) {
  const int64_t k = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  if (k >= n_slices) return;
  const int64_t row = table[2 * k], p0 = table[2 * k + 1];
  if (table[2 * k + 2] <= row) return;  // the row does not end here
  const int64_t a = (int64_t)rowptr[row];
  if (a >= p0) return;  // it begins here
  // slice_table_kernel's rule: the row's first entry lies at or after the slice that starts at
  // or before its position; that slice's piece is empty when its end was rounded down.
  int64_t j = (a + row) / W;
  if (table[2 * j + 3] <= a) ++j;
  const int lane = threadIdx.x & (kWave - 1);
  A acc = A(0);
  for (j += lane; j < k; j += kWave) acc += carry[j];
  acc = wave_sum(acc);
  if (lane == 0) y[row] = T(acc + head[k]);
}

template <typename T, typename A, typename P>
int launch_slices(const void* vals, const int32_t* cols, const void* rowptr, int64_t n_rows,
                  int64_t nnz, const void* x, void* y, int64_t* table, int table_built,
                  void* sums, int cut_rows, hipStream_t st) {
  const int64_t n = slice_count(n_rows, nnz, kSpmvSliceItems);
  const P* rp = static_cast<const P*>(rowptr);
  int rc = FSP_OK;
  if (!table_built)
    rc = launch_slice_table(rowptr, (int)sizeof(P) * 8, n_rows, nnz, kSpmvSliceItems,
                            kSpmvSliceKeep, table, st);
  if (rc) return rc;
  A* carry = static_cast<A*>(sums);
  A* head = carry + n;
  hipLaunchKernelGGL((spmv_slices_kernel<T, A, P>), dim3((unsigned)n), dim3(kBlock), 0, st,
                     static_cast<const T*>(vals), cols, rp, (P)nnz, static_cast<const T*>(x),
                     static_cast<T*>(y), table, carry, head);
  rc = check_hip(hipGetLastError(), "spmv_slices_kernel launch");
  if (rc || !cut_rows) return rc;
  hipLaunchKernelGGL((spmv_slice_fixup_kernel<T, A, P>),
                     dim3((unsigned)((n + kWavesPerBlock - 1) / kWavesPerBlock)), dim3(kBlock), 0,
                     st, rp, table, n, kSpmvSliceItems, carry, head, static_cast<T*>(y));
  return check_hip(hipGetLastError(), "spmv_slice_fixup_kernel launch");
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

int64_t slice_count(int64_t n_rows, int64_t nnz, int64_t W) { return (n_rows + nnz + W - 1) / W; }

int launch_slice_table(const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                       int64_t W, int64_t T, int64_t* table, hipStream_t st) {
  const int64_t n = slice_count(n_rows, nnz, W);
  const unsigned blocks = (unsigned)(n / (kBlock / kProbe) + 1);
  if (rowptr_bits == 32)
    hipLaunchKernelGGL((slice_table_kernel<int>), dim3(blocks), dim3(kBlock), 0, st,
                       static_cast<const int*>(rowptr), n_rows, nnz, W, T, n, table);
  else
    hipLaunchKernelGGL((slice_table_kernel<int64_t>), dim3(blocks), dim3(kBlock), 0, st,
                       static_cast<const int64_t*>(rowptr), n_rows, nnz, W, T, n, table);
  return check_hip(hipGetLastError(), "slice_table_kernel launch");
}

}  // namespace fsp

using namespace fsp;

extern "C" int64_t fsp_slice_order_scratch(int64_t n_slices) {
  if (n_slices < 0) return 0;
  const int64_t tile = order_tile(n_slices);
  return kBins * ((n_slices + tile - 1) / tile);
}

extern "C" int fsp_slice_order(const int64_t* table, int64_t n_slices, const int32_t* cols,
                               int64_t n_cols, int32_t* order, int32_t* scratch, void* stream) {
  if (n_slices < 0 || n_slices > 0x7fffffffLL || n_cols < 1)
    return set_error(FSP_EINVAL, "fsp_slice_order: size out of range");
  if (n_slices == 0) return FSP_OK;
  if (!table || !cols || !order || !scratch)
    return set_error(FSP_EINVAL, "fsp_slice_order: null pointer");
  return launch_order(Slices{table, cols, n_cols, order}, n_slices, scratch,
                      static_cast<hipStream_t>(stream));
}

extern "C" int fsp_part_order(const int32_t* desc, int64_t n_desc, const void* rowptr,
                              int rowptr_bits, int64_t chunk, const int32_t* cols, int64_t n_cols,
                              int32_t* out, int32_t* scratch, void* stream) {
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_part_order: rowptr_bits must be 32 or 64");
  if (n_desc < 0 || n_desc > 0x7fffffffLL || n_cols < 1 || chunk < 1)
    return set_error(FSP_EINVAL, "fsp_part_order: size out of range");
  if (n_desc == 0) return FSP_OK;
  if (!desc || !rowptr || !cols || !out || !scratch || desc == out)
    return set_error(FSP_EINVAL, "fsp_part_order: null pointer, or out is desc");
  if (!aligned16(desc) || !aligned16(out))
    return set_error(FSP_EINVAL, "fsp_part_order: desc and out must be 16-byte aligned");
  const i32x4* d = reinterpret_cast<const i32x4*>(desc);
  i32x4* o = reinterpret_cast<i32x4*>(out);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (rowptr_bits == 32)
    return launch_order(Descriptors<int>{d, static_cast<const int*>(rowptr), chunk, cols, n_cols, o},
                        n_desc, scratch, st);
  return launch_order(
      Descriptors<int64_t>{d, static_cast<const int64_t*>(rowptr), chunk, cols, n_cols, o}, n_desc,
      scratch, st);
}

extern "C" int fsp_slice_pieces(const void* rowptr, int rowptr_bits, int64_t n_slices,
                                int64_t* table, void* stream) {
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_slice_pieces: rowptr_bits must be 32 or 64");
  if (n_slices < 0 || n_slices > 0x3fffffffLL)  // two pieces a slice in 32 bits
    return set_error(FSP_EINVAL, "fsp_slice_pieces: size out of range");
  if (!rowptr || !table) return set_error(FSP_EINVAL, "fsp_slice_pieces: null pointer");
  int* counts = reinterpret_cast<int*>(table + 2 * (n_slices + 1));
  const dim3 grid((unsigned)(n_slices / kBlock + 1));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (rowptr_bits == 32)
    hipLaunchKernelGGL((slice_piece_count_kernel<int>), grid, dim3(kBlock), 0, st,
                       static_cast<const int*>(rowptr), table, n_slices, counts);
  else
    hipLaunchKernelGGL((slice_piece_count_kernel<int64_t>), grid, dim3(kBlock), 0, st,
                       static_cast<const int64_t*>(rowptr), table, n_slices, counts);
  const int rc = check_hip(hipGetLastError(), "slice_piece_count_kernel launch");
  if (rc) return rc;
  hipLaunchKernelGGL(order_scan_kernel, dim3(1), dim3(1024), 0, st, counts, n_slices + 1);
  return check_hip(hipGetLastError(), "order_scan_kernel launch");
}

extern "C" int64_t fsp_spmv_slices(int64_t n_rows, int64_t nnz) {
  return slice_count(n_rows, nnz, kSpmvSliceItems);
}

extern "C" int64_t fsp_spmv_slice_keep(void) { return kSpmvSliceKeep; }
extern "C" int64_t fsp_spmv_slice_items(void) { return kSpmvSliceItems; }

extern "C" int fsp_spmv_sliced(int dtype, int acc_f64, const void* vals, const int32_t* cols,
                               const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                               const void* x, void* y, int64_t* table, int table_built,
                               void* sums, int cut_rows, void* stream) {
  if (dtype != FSP_F32 && dtype != FSP_F64)
    return set_error(FSP_ENOTSUP, "fsp_spmv_sliced: dtype");
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: rowptr_bits must be 32 or 64");
  if (n_rows < 0 || nnz < 0) return set_error(FSP_EINVAL, "fsp_spmv_sliced: negative size");
  if (n_rows > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: more than 2^31-1 rows");
  if (slice_count(n_rows, nnz, kSpmvSliceItems) > kMaxBlocks)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: more slices than a launch holds");
  if (rowptr_bits == 32 && nnz > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: nnz exceeds int32 rowptr range");
  if (n_rows == 0) return FSP_OK;
  if (!rowptr || !y || !table || !sums || (nnz > 0 && (!vals || !cols || !x)))
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: null pointer");
  if (!aligned16(vals) || !aligned16(cols))
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: vals and cols must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define FSP_SLICE_ARGS vals, cols, rowptr, n_rows, nnz, x, y, table, table_built, sums, cut_rows, st
#define FSP_SLICE_CALL(TT, AA)                                                        \
  return rowptr_bits == 32 ? launch_slices<TT, AA, int>(FSP_SLICE_ARGS)                \
                           : launch_slices<TT, AA, int64_t>(FSP_SLICE_ARGS)
  if (dtype == FSP_F64) FSP_SLICE_CALL(double, double);
  if (acc_f64) FSP_SLICE_CALL(float, double);
  FSP_SLICE_CALL(float, float);
#undef FSP_SLICE_CALL
#undef FSP_SLICE_ARGS
}
