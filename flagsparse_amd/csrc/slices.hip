// CSR SpMV without a plan: the matrix cut into slices of about equal work, for calls that use
// a matrix once (no prepared object).
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
// row there by binary search.  A boundary inside a row of at most T entries moves to that row's
// start, so only longer rows are cut; a slice holds at most W + T + 3 rows and entries
// together, whatever the row lengths, empty rows included.
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

template <typename P>
__global__ __launch_bounds__(kBlock) void slice_table_kernel(const P* __restrict__ rowptr,
                                                             int64_t n_rows, int64_t nnz,
                                                             int64_t W, int64_t T,
                                                             int64_t n_slices,
                                                             int64_t* __restrict__ table) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k > n_slices) return;
  int64_t row = n_rows, pos = nnz;
  if (k < n_slices) {
    const int64_t d = k * W;  // < n_rows + nnz
    int64_t lo = 0, hi = n_rows;  // the largest i with rowptr[i] + i <= d (true for i = 0)
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo + 1) / 2;
      if ((int64_t)rowptr[mid] + mid <= d) lo = mid;
      else hi = mid - 1;
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
  table[2 * k] = row;
  table[2 * k + 1] = pos;
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
    const P base = s0 + P(4) * (tid + u * kBlock);
    if (base < p1) {
      QuadLoader<false, T>::load(vals, cols, base, p0, p1, nnz_total, v[u], c[u]);
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
    const P base = s0 + P(4) * (tid + u * kBlock);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (c[u][j] >= 0) s_prod[(int)(base + j - p0)] = A(v[u][j]) * A(xv[u][j]);
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
                  int64_t nnz, const void* x, void* y, int64_t* table, void* sums, int cut_rows,
                  hipStream_t st) {
  const int64_t n = slice_count(n_rows, nnz, kSpmvSliceItems);
  const P* rp = static_cast<const P*>(rowptr);
  int rc = launch_slice_table(rowptr, (int)sizeof(P) * 8, n_rows, nnz, kSpmvSliceItems,
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
  const unsigned blocks = (unsigned)(n / kBlock + 1);
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

extern "C" int64_t fsp_spmv_slices(int64_t n_rows, int64_t nnz) {
  return slice_count(n_rows, nnz, kSpmvSliceItems);
}

extern "C" int64_t fsp_spmv_slice_keep(void) { return kSpmvSliceKeep; }

extern "C" int fsp_spmv_sliced(int dtype, int acc_f64, const void* vals, const int32_t* cols,
                               const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                               const void* x, void* y, int64_t* table, void* sums, int cut_rows,
                               void* stream) {
  if (dtype != FSP_F32 && dtype != FSP_F64)
    return set_error(FSP_ENOTSUP, "fsp_spmv_sliced: dtype");
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: rowptr_bits must be 32 or 64");
  if (n_rows < 0 || nnz < 0) return set_error(FSP_EINVAL, "fsp_spmv_sliced: negative size");
  if (n_rows > 0x7fffffffLL || slice_count(n_rows, nnz, kSpmvSliceItems) > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: more than 2^31-1 rows or slices");
  if (rowptr_bits == 32 && nnz > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: nnz exceeds int32 rowptr range");
  if (n_rows == 0) return FSP_OK;
  if (!rowptr || !y || !table || !sums || (nnz > 0 && (!vals || !cols || !x)))
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: null pointer");
  if (!aligned16(vals) || !aligned16(cols))
    return set_error(FSP_EINVAL, "fsp_spmv_sliced: vals and cols must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define FSP_SLICE_ARGS vals, cols, rowptr, n_rows, nnz, x, y, table, sums, cut_rows, st
#define FSP_SLICE_CALL(TT, AA)                                                        \
  return rowptr_bits == 32 ? launch_slices<TT, AA, int>(FSP_SLICE_ARGS)                \
                           : launch_slices<TT, AA, int64_t>(FSP_SLICE_ARGS)
  if (dtype == FSP_F64) FSP_SLICE_CALL(double, double);
  if (acc_f64) FSP_SLICE_CALL(float, double);
  FSP_SLICE_CALL(float, float);
#undef FSP_SLICE_CALL
#undef FSP_SLICE_ARGS
}
