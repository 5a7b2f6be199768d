// CSR SDDMM over slices of equal work: out[p] = alpha * dot(x[row(p)], y[col(p)]) + beta * in[p].
//
// Reference behaviour followed: as sddmm.hip (sddmm_csr.py:107-151, 271-347).
//
// The slices are those of slices.hip with every boundary where it falls (entries are
// independent, so a cut row has no pieces to add).  A workgroup stages its slice's columns in
// LDS and gives each of its groups of G lanes the same number of consecutive entries, whatever
// rows they lie in: the group finds its first row by binary search in LDS, keeps that row of x in
// registers (VW consecutive elements a lane and step, KC steps) and takes up to four of the row's
// entries at a time.  Results are collected in LDS and written out in whole lines.
//   * VW is 4 (float32) or 2 (float64) for every K that holds a vector, at any alignment; when K
//     is no whole number of vectors, the lane that reaches past K moves back to end there and
//     drops the elements its neighbour has (ragged).
//   * a step's positions past a row's end read y's first row, which stays in the cache: with one
//     or two entries to a row, reading the last entry again cost as much as an entry each.
//
// Bound: the y rows' fills from outside L2 (whole 128-byte lines), as sddmm_rowblock_kernel.
// Measured on MI355X, row blocks / slices: fp32 K=64, 33.5M entries 684 / 676 us; K=33, 1.6M
// entries in rows of 0 to 32 60.8 / 50.7; fp64 K=50, a power law of 1M 90 / 68; K=7, 3M 44.6 /
// 25.4.  Elements dropped by a test on every product instead of the three fits: fp32 K=64 690.
#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

// The row pointers at either width: read once per row of a slice.
__device__ __forceinline__ int64_t row_start(const void* rowptr, int bits, int64_t r) {
  return bits == 32 ? (int64_t) static_cast<const int32_t*>(rowptr)[r]
                    : static_cast<const int64_t*>(rowptr)[r];
}

// How a lane's vectors lie in a row: every one inside it (K = KC * G * VW), some past its end, or
// one reaching past it as well.
enum { kExact, kWhole, kRagged };

template <typename T, typename A, typename O, int VW, int KC, int FIT>
__global__ __launch_bounds__(kBlock) void sddmm_slices_kernel(
    const int* __restrict__ cols, const void* __restrict__ rowptr, int rowptr_bits,
    int64_t nnz_total, const T* __restrict__ x, int64_t ldx, const T* __restrict__ y,
    uint32_t ldy, int K, const T* __restrict__ in, double alpha, double beta,
    O* __restrict__ out, const int64_t* __restrict__ table, const int* __restrict__ order,
    int n_slices, int cap, int rows_cap, int lg) {
  extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
  // s_out [cap] (a 4-byte result takes its column's slot) | s_col [cap] | s_ptr [rows_cap + 2]
  constexpr bool kShared = sizeof(O) == sizeof(int);
  O* s_out = reinterpret_cast<O*>(s_raw);
  int* s_col = kShared ? reinterpret_cast<int*>(s_raw) : reinterpret_cast<int*>(s_out + cap);
  int* s_ptr = s_col + cap;
  const int G = 1 << lg, ngrp = kBlock >> lg;

  const int tid = threadIdx.x;
  const int64_t k = order ? order[blockIdx.x] : xcd_logical_block(blockIdx.x, n_slices);
  const int grp = tid >> lg, lane = tid & (G - 1);
  const int64_t i0 = table[2 * k], p0 = table[2 * k + 1];
  const int64_t i1 = table[2 * k + 2], p1 = table[2 * k + 3];
  if (i1 < i0 || i1 - i0 > rows_cap || p1 < p0 || p1 - p0 > cap - 3) return;  // uniform
  const int R = (int)(i1 - i0), n = (int)(p1 - p0);
  {
    const int64_t s0 = p0 & ~int64_t(3);
    for (int64_t base = s0 + 4 * tid; base < p1; base += 4 * kBlock) {
      int cc[4];
      if (base + 4 <= nnz_total) {
        const i32x4 v = *reinterpret_cast<const i32x4*>(cols + base);
        cc[0] = v.x; cc[1] = v.y; cc[2] = v.z; cc[3] = v.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) cc[j] = base + j < nnz_total ? cols[base + j] : 0;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (base + j >= p0 && base + j < p1) s_col[(int)(base + j - p0)] = cc[j];
    }
    for (int s = tid; s <= R; s += kBlock) {
      const int64_t a = row_start(rowptr, rowptr_bits, i0 + s);
      s_ptr[s] = a > p0 ? (int)(a - p0) : 0;
    }
    if (tid == 0) s_ptr[R + 1] = n;
  }
  __syncthreads();

  // This lane's elements of a row: step c covers [kb[c], kb[c] + VW), of which the first drop[c]
  // belong to the lane before; a step past K reads element 0 and is dropped.
  int kb[KC], drop[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    const int k0 = (lane + c * G) * VW;
    kb[c] = k0;
    drop[c] = 0;
    if (k0 >= K) {
      kb[c] = 0;
      drop[c] = VW;
    } else if (FIT == kRagged && k0 + VW > K) {
      kb[c] = K - VW;  // K >= VW (host check)
      drop[c] = k0 - kb[c];
    }
  }
  auto dropped = [&](int c, int j) {
    if constexpr (FIT == kExact) return false;
    else if constexpr (FIT == kWhole) return drop[c] != 0;
    else return j < drop[c];
  };
  const A a_alpha = A(alpha), a_beta = A(beta);
  const int each = ((n + ngrp - 1) / ngrp + 3) & ~3;
  int i = grp * each;
  const int end = i + each < n ? i + each : n;
  int s = 0, row_end = 0;
  if (i < end) {
    int hi = R;  // the last row of the slice that starts at or before entry i (row 0 does)
    while (s < hi) {
      const int mid = (s + hi + 1) >> 1;
      if (s_ptr[mid] <= i) s = mid;
      else hi = mid - 1;
    }
  }
  T xr[KC][VW];
#pragma unroll 1
  while (i < end) {
    if (i >= row_end) {  // the first row, or the next one that has entries
      while (s_ptr[s + 1] <= i) ++s;
      row_end = s_ptr[s + 1];
      const T* xp = x + (i0 + s) * ldx;
#pragma unroll
      for (int c = 0; c < KC; ++c) load_any<T, VW>(xp + kb[c], xr[c]);
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < VW; ++j)
          if (dropped(c, j)) xr[c][j] = T(0);
    }
    const int e = row_end < end ? row_end : end;
    T yv[4][KC][VW];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const T* yp = y + (uint64_t)(i + q < e ? (uint32_t)s_col[i + q] : 0u) * ldy;
#pragma unroll
      for (int c = 0; c < KC; ++c) load_any<T, VW>(yp + kb[c], yv[q][c]);
    }
    __builtin_amdgcn_sched_barrier(0);  // all requested before the first is waited for
    A acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // A vector's products in a chain of fused steps, which rounds one product where pairs would
      // round two; then vectors, then lanes: no running sum is longer than a vector, so fewer
      // lanes (more steps) lose no precision.  Error against 64 bits, in 1e-8 of the result's norm,
      // row blocks / pairs / so: fp32 K=8 4.829 / 4.920 / 4.829, K=64 6.766 / 6.832 / 6.766, K=256
      // 9.61 / 7.84 / 7.78.  A dropped element is 0 in both rows (an infinity or a NaN next to 0
      // would show).
      A part[KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        A a[VW], b[VW];
#pragma unroll
        for (int j = 0; j < VW; ++j) {
          a[j] = A(xr[c][j]);
          b[j] = A(dropped(c, j) ? T(0) : yv[q][c][j]);
        }
        if constexpr (VW == 1) part[c] = a[0] * b[0];
        else if constexpr (VW == 2) part[c] = fma(a[1], b[1], a[0] * b[0]);
        else part[c] = fma(a[3], b[3], fma(a[2], b[2], fma(a[1], b[1], a[0] * b[0])));
      }
      if constexpr (KC == 1) acc[q] = part[0];
      else if constexpr (KC == 2) acc[q] = part[0] + part[1];
      else acc[q] = (part[0] + part[1]) + (part[2] + part[3]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = group_sum(acc[q], G);
    // Every lane of the group holds the four sums; a slot's column was read above by this group
    // only, so its result may take the slot (the group's lanes run in lockstep).
    if (G >= 4) {
      if (lane < 4 && i + lane < e) {
        A v = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
        v *= a_alpha;
        if (in) v += A(in[p0 + i + lane]) * a_beta;
        s_out[i + lane] = O(v);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if ((q & (G - 1)) == lane && i + q < e) {
          A v = acc[q] * a_alpha;
          if (in) v += A(in[p0 + i + q]) * a_beta;
          s_out[i + q] = O(v);
        }
      }
    }
    i = i + 4 < e ? i + 4 : e;
  }
  __syncthreads();
  for (int i = tid; i < n; i += kBlock) out[p0 + i] = s_out[i];
}

struct SdArgs {
  const int32_t* cols;
  const void* rowptr;
  int rowptr_bits;
  int64_t n_rows, nnz;
  const void* x;
  int64_t ldx;
  const void* y;
  int64_t ldy, K;
  const void* in;
  double alpha, beta;
  void* out;
  const int64_t* table;
  const int32_t* order;
  int64_t items;
  int lg;
  hipStream_t st;
};

template <typename T, typename A, typename O, int VW, int KC, int FIT>
int launch_sd(const SdArgs& a) {
  const int64_t n = slice_count(a.n_rows, a.nnz, a.items);
  const int cap = (int)((a.items + 6 + 3) & ~int64_t(3));
  const int rows_cap = (int)a.items + 3;
  const size_t lds = (size_t)cap * (sizeof(O) == 4 ? 4 : sizeof(O) + 4) +
                     4 * (size_t)(rows_cap + 2);
  hipLaunchKernelGGL((sddmm_slices_kernel<T, A, O, VW, KC, FIT>), dim3((unsigned)n),
                     dim3(kBlock), lds, a.st, a.cols, a.rowptr, a.rowptr_bits, a.nnz,
                     static_cast<const T*>(a.x), a.ldx, static_cast<const T*>(a.y),
                     (uint32_t)a.ldy, (int)a.K, static_cast<const T*>(a.in), a.alpha, a.beta,
                     static_cast<O*>(a.out), a.table, a.order, (int)n, cap, rows_cap, a.lg);
  return check_hip(hipGetLastError(), "sddmm_slices_kernel launch");
}

template <typename T, typename A, typename O, int VW>
int launch_kc(const SdArgs& a) {
  const int64_t per = (int64_t)VW << a.lg;
  const int kc = (int)((a.K + per - 1) / per);
#define FSP_SD(KCV)                                                                     \
  do {                                                                                  \
    if (a.K == KCV * per) return launch_sd<T, A, O, VW, KCV, kExact>(a);                \
    if constexpr (VW > 1) {                                                             \
      if (a.K % VW != 0) return launch_sd<T, A, O, VW, KCV, kRagged>(a);                \
    }                                                                                   \
    return launch_sd<T, A, O, VW, KCV, kWhole>(a);                                      \
  } while (0)
  if (kc <= 1) FSP_SD(1);
  if (kc <= 2) FSP_SD(2);
  FSP_SD(4);
#undef FSP_SD
}

template <typename T, typename A, typename O>
int launch_vec(const SdArgs& a, int vec) {
  if constexpr (sizeof(T) == 4) {
    if (vec == 4) return launch_kc<T, A, O, 4>(a);
  }
  if (vec == 2) return launch_kc<T, A, O, 2>(a);
  return launch_kc<T, A, O, 1>(a);
}

}  // namespace
}  // namespace fsp

using namespace fsp;

extern "C" int fsp_sddmm_sliced(int dtype, int acc_f64, int out_f64, const int32_t* cols,
                                const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                                const void* x, int64_t ldx, const void* y, int64_t ldy,
                                int64_t K, const void* data_in, double alpha, double beta,
                                void* out, const int64_t* table, const int32_t* order,
                                int64_t items, int lanes_per_entry, int vec, void* stream) {
  if (dtype != FSP_F32 && dtype != FSP_F64)
    return set_error(FSP_ENOTSUP, "fsp_sddmm_sliced: dtype");
  if (nnz < 0 || n_rows < 0 || K < 1)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: negative size or K < 1");
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: rowptr_bits must be 32 or 64");
  if (n_rows > 0x7fffffffLL || ldy > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: size exceeds 2^31-1");
  int lg = -1;
  for (int g = 0; g <= 6; ++g)
    if (lanes_per_entry == (1 << g)) lg = g;
  if (lg < 0)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: lanes_per_entry must be 1,2,4,...,64");
  const int max_vec = dtype == FSP_F32 ? 4 : 2;
  if (vec != 1 && vec != 2 && vec != max_vec)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: vec must be 1, 2 or 4 (fp32) / 1, 2 (fp64)");
  if (K < vec || K > 4 * ((int64_t)vec << lg))
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: needs vec <= K <= 4 * lanes * vec");
  if (items < 1 || items > 2048)  // 33 KB of LDS with float64 results
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: items outside [1, 2048]");
  if (ldx < K || ldy < K)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: ldx/ldy smaller than K");
  if (out_f64 && dtype != FSP_F32)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: out_f64 applies to fp32 inputs only");
  if (slice_count(n_rows, nnz, items) > kMaxBlocks)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: more slices than a launch holds");
  if (nnz == 0) return FSP_OK;
  if (!cols || !rowptr || !x || !y || !out || !table)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: null pointer");
  if (reinterpret_cast<uintptr_t>(cols) % 16)
    return set_error(FSP_EINVAL, "fsp_sddmm_sliced: cols must be 16-byte aligned");
  const SdArgs a{cols, rowptr, rowptr_bits, n_rows, nnz,   x,    ldx,  y,     ldy,
                 K,    data_in, alpha,      beta,   out,   table, order, items, lg,
                 static_cast<hipStream_t>(stream)};
  if (dtype == FSP_F64) return launch_vec<double, double, double>(a, vec);
  if (out_f64) return launch_vec<float, double, double>(a, vec);
  if (acc_f64) return launch_vec<float, double, float>(a, vec);
  return launch_vec<float, float, float>(a, vec);
}
