// CSR SpMM C = A @ B over slices of equal work (row-major B and C): no plan, and blocks that
// stay full whatever the row lengths.
//
// Reference behaviour followed: as spmm.hip (spmm_csr.py:92-134, 602-919).
//
// The slices are those of slices.hip: W positions (rows + entries) each, boundaries moved to a
// row start unless the row has more than T entries.  W grows with the lane groups a workgroup
// holds (slice_shape in spmm_csr.py), so that a group has several entries whether the slice
// holds sixteen rows of 32 entries or a hundred of three; a row-block plan with one row per
// group leaves such short rows in workgroups that are mostly latency.
//   * G lanes share one B row, VW consecutive columns each.  VW is 4 (float32) or 2 (float64)
//     for every N that holds a vector: gfx950 loads 16 bytes from any element's address, so an
//     odd N needs no narrow lanes.  The group's last lane moves back to end at column N; the
//     columns it shares with its neighbour come out the same in both.
//   * the slice's (column, value) entries are staged in LDS with 16-byte loads; group g takes
//     the slice's rows g, g + ngrp, ... alone, U B rows in flight per lane, the last few entries
//     of a row in one masked step instead of one by one.
//   * a row much longer than the groups' share of the slice is left to a second step, where all
//     groups take its entries in turn and their sums are added through LDS in a fixed order.
//   * the piece of a row that goes on in the next slice goes to carry[k], the end of a row begun
//     earlier to head[k]; spmm_slice_fixup_kernel adds the pieces in slice order.  A slot for either
//     of every slice needs no count; where that is much room (wide N, few cut rows), the pieces are
//     counted (fsp_slice_pieces) and lie one after the other: slice k's from pieces[k] (COUNTED,
//     a kernel of its own: as a test in the other it cost single elements 13 %, 50k rows of 200,
//     fp32 N=3 33.5 / 38.1 us).
//
// Bound: the B rows' fills from outside L2 (whole 128-byte lines), as spmm_rowblock_kernel.
// Measured on MI355X, row blocks / slices: a power law of 200k rows and 4.8M entries, fp32 N=47
// 326.5 / 214 us (kernel 229 / 206: 188-byte rows span 2.5 lines on average, 1.5 GB of fills; the
// second pass 94 / 8); 300k rows, N=128 457 / 316 us; 3M entries, N=33 80.6 / 53.0 us.
#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

constexpr int kInFlight = 4;  // B rows requested together per lane

// acc += the products of entries a, a + step, ... < e of the staged slice.
template <typename T, typename A, int VW>
__device__ __forceinline__ void add_entries(const int* s_col, const T* s_val, int a, int e,
                                            int step, const T* Bc, uint32_t ldb, A (&acc)[VW]) {
  int i = a;
  for (; i + (kInFlight - 1) * step < e; i += kInFlight * step) {
    T bv[kInFlight][VW];
#pragma unroll
    for (int q = 0; q < kInFlight; ++q)
      load_any<T, VW>(Bc + (uint64_t)(uint32_t)s_col[i + q * step] * ldb, bv[q]);
    __builtin_amdgcn_sched_barrier(0);  // all requested before the first is waited for
#pragma unroll
    for (int q = 0; q < kInFlight; ++q) {
      const A av = A(s_val[i + q * step]);
#pragma unroll
      for (int j = 0; j < VW; ++j) acc[j] += av * A(bv[q][j]);
    }
  }
  if (i < e) {
    // The rest in one step: a position past the end reads B's first row, which stays in the
    // cache, and the value is dropped (not multiplied by 0: it may be an infinity or a NaN).
    T bv[kInFlight - 1][VW];
#pragma unroll
    for (int q = 0; q < kInFlight - 1; ++q) {
      const bool use = i + q * step < e;
      load_any<T, VW>(Bc + (uint64_t)(use ? (uint32_t)s_col[i + q * step] : 0u) * ldb, bv[q]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kInFlight - 1; ++q) {
      const bool use = i + q * step < e;
      const A av = use ? A(s_val[i + q * step]) : A(0);
#pragma unroll
      for (int j = 0; j < VW; ++j) acc[j] += av * A(use ? bv[q][j] : T(0));
    }
  }
}

// UPT: quads of entries per thread (a slice holds at most UPT * 1024 - 3 entries).
template <typename T, typename A, typename P, int VW, int UPT, bool COUNTED>
__global__ __launch_bounds__(kBlock, 8) void spmm_slices_kernel(
    const T* __restrict__ vals, const int* __restrict__ cols, const P* __restrict__ rowptr,
    P nnz_total, const T* __restrict__ B, uint32_t ldb, int N, T* __restrict__ C, int64_t ldc,
    const int64_t* __restrict__ table, const int* __restrict__ order, int n_slices, int cap,
    int rows_cap, int lg, A* __restrict__ carry, A* __restrict__ head,
    const int* __restrict__ pieces, int xcd_remap) {
  extern __shared__ __attribute__((aligned(16))) unsigned char s_raw[];
  // s_red [4 waves][G * VW] | s_val [cap] | s_col [cap] | s_ptr [rows_cap + 2] | s_list | s_n
  const int G = 1 << lg, ngrp = kBlock >> lg, W = G * VW;
  A* s_red = reinterpret_cast<A*>(s_raw);
  T* s_val = reinterpret_cast<T*>(s_red + kWavesPerBlock * W);
  int* s_col = reinterpret_cast<int*>(s_val + cap);
  int* s_ptr = s_col + cap;
  int* s_list = s_ptr + rows_cap + 2;
  int* s_n = s_list + ngrp;

  const int tid = threadIdx.x;
  int k = blockIdx.x;
  if (order) k = order[k];
  else if (xcd_remap) k = xcd_logical_block(k, n_slices);
  const int tile = blockIdx.y;
  const int grp = tid >> lg, lane = tid & (G - 1);
  const int64_t i0 = table[2 * (int64_t)k], i1 = table[2 * (int64_t)k + 2];
  const P p0 = (P)table[2 * (int64_t)k + 1], p1 = (P)table[2 * (int64_t)k + 3];
  const int64_t R64 = i1 - i0;
  if (R64 < 0 || R64 > rows_cap || p1 < p0 || p1 - p0 > P(cap - 3)) return;  // uniform
  const int R = (int)R64, n = (int)(p1 - p0);
  {
    const P s0 = p0 & ~P(3);
    T v[UPT][4];
    int c[UPT][4];
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const Wide<P> base = Wide<P>(s0) + 4 * (tid + u * kBlock);
      if (base < Wide<P>(p1)) {
        QuadLoader<true, T>::load(vals, cols, P(base), p0, p1, nnz_total, v[u], c[u]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[u][j] = T(0); c[u][j] = -1; }
      }
    }
    for (int s = tid; s <= R; s += kBlock) {
      const P a = rowptr[i0 + s];
      s_ptr[s] = a > p0 ? (int)(a - p0) : 0;
    }
    if (tid == 0) {
      s_ptr[R + 1] = n;
      *s_n = 0;
    }
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const Wide<P> base = Wide<P>(s0) + 4 * (tid + u * kBlock);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c[u][j] >= 0) {
          const int o = (int)(base + j - Wide<P>(p0));
          s_col[o] = c[u][j];
          s_val[o] = v[u][j];
        }
    }
  }
  const bool begun = R > 0 && rowptr[i0] < p0;  // row i0 began in an earlier slice and ends here
  __syncthreads();

  int ncol = tile * W + lane * VW;
  const bool col_ok = ncol < N;
  if (ncol + VW > N) ncol = N >= VW ? N - VW : 0;  // N < VW only with VW == 1 (host check)
  const T* Bc = B + ncol;
  auto put = [&](int s, const A(&acc)[VW]) {
    if (s == R) {
      const int64_t slot = COUNTED ? pieces[k] + (begun ? 1 : 0) : k;
      store_any<A, A, VW>(carry + slot * N + ncol, acc);
    } else if (s == 0 && begun) {
      const int64_t slot = COUNTED ? pieces[k] : k;
      store_any<A, A, VW>(head + slot * N + ncol, acc);
    } else {
      store_any<T, A, VW>(C + (i0 + s) * ldc + ncol, acc);
    }
  };
  // Step 0: where the slice holds fewer rows than there are groups, S groups of a wave share a
  // row (the entries in turn, their sums added by lane exchanges).  Rows longer than twice a
  // share are listed: at most ngrp / 2 of them.
  // Step 1: a listed row of at most a quarter of the slice is one wave's.
  // Step 2: a longer one (at most three) is every wave's, the sums added through LDS.
  int ls = 0;
  while (((ngrp >> ls) >> 1) > R && (G << ls) < kWave) ++ls;
  const int nsg = ngrp >> ls, wgrp = kWave >> lg, wave = tid / kWave;
  const int share = (n + nsg - 1) / nsg;
  const int limit = share > 16 ? 2 * share : 32;
  const int by_wave = (n + kWavesPerBlock - 1) / kWavesPerBlock;
  int count = R + 1, it = grp >> ls, stride = nsg;
  int step = 1 << ls, part = grp & (step - 1), span = G << ls;
#pragma unroll 1
  for (int phase = 0; phase < 3; ++phase) {
#pragma unroll 1
    for (; it < count; it += stride) {
      const int s = phase ? s_list[it] : it;
      const int a = s_ptr[s], e = s_ptr[s + 1];
      if (phase == 0) {
        if (e - a > limit) {
          if (lane == 0 && part == 0) s_list[atomicAdd(s_n, 1)] = s;
          continue;
        }
        if (s == R && e == a) continue;  // no piece of row i1 in this slice
      } else if ((e - a > by_wave) != (phase == 2)) {
        continue;
      }
      A acc[VW];
#pragma unroll
      for (int j = 0; j < VW; ++j) acc[j] = A(0);
      if (col_ok) add_entries<T, A, VW>(s_col, s_val, a + part, e, step, Bc, ldb, acc);
      for (int off = G; off < span; off <<= 1) {
#pragma unroll
        for (int j = 0; j < VW; ++j) acc[j] += __shfl_xor(acc[j], off, kWave);
      }
      bool mine = col_ok && part == 0;
      if (phase == 2) {  // uniform: every thread is here
        if ((grp & (wgrp - 1)) == 0) {
#pragma unroll
          for (int j = 0; j < VW; ++j) s_red[wave * W + lane * VW + j] = acc[j];
        }
        __syncthreads();
        if (mine) {  // the first group of wave 0
#pragma unroll
          for (int w = 1; w < kWavesPerBlock; ++w)
#pragma unroll
            for (int j = 0; j < VW; ++j) acc[j] += s_red[w * W + lane * VW + j];
        }
        __syncthreads();
      }
      if (mine) put(s, acc);
    }
    if (phase == 0) {
      __syncthreads();
      count = *s_n;
      it = wave;
      stride = kWavesPerBlock;
      step = wgrp;
      part = grp & (wgrp - 1);
      span = kWave;
    } else {
      it = 0;
      stride = 1;
      step = ngrp;
      part = grp;
    }
  }
}

// The rows that were cut: C[row, :] = the carries of the slices the row began in and crossed, in
// order, plus the head of the slice it ends in.  A workgroup per slice, most of which have no
// such end: cw threads side by side over the columns, the 256 / cw groups over the pieces, their
// sums added in a fixed tree.  (64 slices to a workgroup: a power law's many rows of a few
// pieces then wait for each other, 32 instead of 8 us at N = 47.)
template <typename T, typename A, typename P, bool COUNTED>
__global__ __launch_bounds__(kBlock) void spmm_slice_fixup_kernel(
    const P* __restrict__ rowptr, const int64_t* __restrict__ table, int64_t Wpos,
    const A* __restrict__ carry, const A* __restrict__ head, const int* __restrict__ pieces, int N,
    int cw, T* __restrict__ C, int64_t ldc) {
  __shared__ A s_red[kBlock];
  const int tid = threadIdx.x;
  const int64_t k = blockIdx.x, row = table[2 * k], p0 = table[2 * k + 1];
  if (table[2 * k + 2] <= row) return;  // the row does not end here
  const int64_t a = (int64_t)rowptr[row];
  if (a >= p0) return;  // it begins here
  int64_t j0 = (a + row) / Wpos;  // the slice the row began in (spmv_slice_fixup_kernel)
  if (table[2 * j0 + 3] <= a) ++j0;
  if constexpr (COUNTED) {  // the row's pieces lie one after the other, up to pieces[k]
    carry += (pieces[k] - k) * N;
    head += (pieces[k] - k) * N;
  }
  const int c0 = tid & (cw - 1), pg = tid / cw, npg = kBlock / cw;
  for (int cb = 0; cb < N; cb += cw) {
    const int c = cb + c0;
    A acc = A(0);
    if (c < N) {
      int64_t j = j0 + pg;
      for (; j + 7 * npg < k; j += 8 * npg) {
        A t[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) t[q] = carry[(j + q * npg) * N + c];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += t[q];
      }
      for (; j < k; j += npg) acc += carry[j * N + c];
    }
    s_red[tid] = acc;
    __syncthreads();
    for (int h = npg / 2; h >= 1; h >>= 1) {
      if (pg < h) s_red[tid] += s_red[tid + h * cw];
      __syncthreads();
    }
    if (pg == 0 && c < N) C[row * ldc + c] = T(s_red[c0] + head[k * N + c]);
    __syncthreads();
  }
}

struct SliceArgs {
  const void* vals;
  const int32_t* cols;
  const void* rowptr;
  int64_t n_rows, nnz;
  const void* B;
  int64_t ldb, N;
  void* C;
  int64_t ldc;
  const int64_t* table;
  const int32_t* order;
  void* sums;
  int64_t items, keep;
  int cut_rows, lg, xcd_remap;
  hipStream_t st;
};

template <typename T, typename A, typename P, int VW, int UPT, bool COUNTED>
int launch_upt(const SliceArgs& a) {
  const int64_t n = slice_count(a.n_rows, a.nnz, a.items);
  const int cap = (int)((a.items + a.keep + 6 + 3) & ~int64_t(3));
  const int rows_cap = (int)(a.items + a.keep + 3);
  const int W = VW << a.lg;
  const int64_t tiles = (a.N + W - 1) / W;
  const size_t lds = (size_t)kWavesPerBlock * W * sizeof(A) + (size_t)cap * (sizeof(T) + 4) +
                     4 * (size_t)(rows_cap + 2 + (kBlock >> a.lg) + 1);
  A* carry = static_cast<A*>(a.sums);
  A* head = COUNTED ? carry : carry + n * a.N;
  const int* pieces = COUNTED ? reinterpret_cast<const int*>(a.table + 2 * (n + 1)) : nullptr;
  hipLaunchKernelGGL((spmm_slices_kernel<T, A, P, VW, UPT, COUNTED>),
                     dim3((unsigned)n, (unsigned)tiles), dim3(kBlock), lds, a.st,
                     static_cast<const T*>(a.vals), a.cols, static_cast<const P*>(a.rowptr),
                     (P)a.nnz, static_cast<const T*>(a.B), (uint32_t)a.ldb, (int)a.N,
                     static_cast<T*>(a.C), a.ldc, a.table, a.order, (int)n, cap, rows_cap, a.lg,
                     carry, head, pieces, a.xcd_remap);
  int rc = check_hip(hipGetLastError(), "spmm_slices_kernel launch");
  if (rc || !a.cut_rows) return rc;
  int cw = 1;
  while (cw < a.N && cw < kBlock) cw <<= 1;
  hipLaunchKernelGGL((spmm_slice_fixup_kernel<T, A, P, COUNTED>), dim3((unsigned)n),
                     dim3(kBlock), 0, a.st, static_cast<const P*>(a.rowptr), a.table, a.items,
                     carry, head, pieces, (int)a.N, cw, static_cast<T*>(a.C), a.ldc);
  return check_hip(hipGetLastError(), "spmm_slice_fixup_kernel launch");
}

template <typename T, typename A, typename P, int VW>
int launch_vec(const SliceArgs& a) {
  const bool counted = a.cut_rows == FSP_CUT_PIECES;
  if (a.items + a.keep + 6 <= 4 * kBlock)
    return counted ? launch_upt<T, A, P, VW, 1, true>(a) : launch_upt<T, A, P, VW, 1, false>(a);
  return counted ? launch_upt<T, A, P, VW, 2, true>(a) : launch_upt<T, A, P, VW, 2, false>(a);
}

template <typename T, typename A, typename P>
int launch_ptr(const SliceArgs& a, int vec) {
  if constexpr (sizeof(T) == 4) {
    if (vec == 4) return launch_vec<T, A, P, 4>(a);
  }
  if (vec == 2) return launch_vec<T, A, P, 2>(a);
  return launch_vec<T, A, P, 1>(a);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace fsp

using namespace fsp;

extern "C" int64_t fsp_slice_count(int64_t n_rows, int64_t nnz, int64_t items) {
  return items > 0 ? slice_count(n_rows, nnz, items) : 0;
}

extern "C" int fsp_slice_table(const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                               int64_t items, int64_t keep, int64_t* table, void* stream) {
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_slice_table: rowptr_bits must be 32 or 64");
  if (n_rows < 0 || nnz < 0 || items < 1 || keep < 0)
    return set_error(FSP_EINVAL, "fsp_slice_table: bad size");
  if (slice_count(n_rows, nnz, items) > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_slice_table: more than 2^31-1 slices");
  if (!rowptr || !table) return set_error(FSP_EINVAL, "fsp_slice_table: null pointer");
  return launch_slice_table(rowptr, rowptr_bits, n_rows, nnz, items, keep, table,
                            static_cast<hipStream_t>(stream));
}

extern "C" int fsp_spmm_sliced(int dtype, int acc_f64, const void* vals, const int32_t* cols,
                               const void* rowptr, int rowptr_bits, int64_t n_rows, int64_t nnz,
                               const void* B, int64_t ldb, int64_t N, void* C, int64_t ldc,
                               const int64_t* table, const int32_t* order, int64_t items,
                               int64_t keep, void* sums, int cut_rows, int lanes_per_row, int vec, int xcd_remap,
                               void* stream) {
  if (dtype != FSP_F32 && dtype != FSP_F64)
    return set_error(FSP_ENOTSUP, "fsp_spmm_sliced: dtype");
  if (rowptr_bits != 32 && rowptr_bits != 64)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: rowptr_bits must be 32 or 64");
  if (n_rows < 0 || nnz < 0 || N < 0)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: negative size");
  if (n_rows > 0x7fffffffLL || N > 0x7fffffffLL || ldb > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: size exceeds 2^31-1");
  if (rowptr_bits == 32 && nnz > 0x7fffffffLL)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: nnz exceeds int32 rowptr range");
  if (items < 1 || keep < 0 || items > 8 * kBlock || items + keep + 6 > 8 * kBlock)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: a slice must hold at most 2042 positions");
  int lg = -1;
  for (int g = 0; g <= 6; ++g)
    if (lanes_per_row == (1 << g)) lg = g;
  if (lg < 0) return set_error(FSP_EINVAL, "fsp_spmm_sliced: lanes_per_row must be 1,2,4,...,64");
  const int max_vec = dtype == FSP_F32 ? 4 : 2;
  if (vec != 1 && vec != 2 && vec != max_vec)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: vec must be 1, 2 or 4 (fp32) / 1, 2 (fp64)");
  if (n_rows == 0 || N == 0) return FSP_OK;
  if (N < vec) return set_error(FSP_EINVAL, "fsp_spmm_sliced: N smaller than vec");
  if (ldb < N || ldc < N)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: ldb/ldc smaller than N");
  if (!rowptr || !C || !table || (nnz > 0 && (!vals || !cols || !B)))
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: null pointer");
  if (cut_rows && !sums) return set_error(FSP_EINVAL, "fsp_spmm_sliced: null sums");
  if (!aligned16(vals) || !aligned16(cols) || !aligned16(sums))
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: vals, cols and sums must be 16-byte aligned");
  const int64_t W = (int64_t)lanes_per_row * vec;
  if ((N + W - 1) / W > 65535)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: too many column tiles");
  if (slice_count(n_rows, nnz, items) > kMaxBlocks)
    return set_error(FSP_EINVAL, "fsp_spmm_sliced: more slices than a launch holds");
  const SliceArgs a{vals, cols, rowptr, n_rows, nnz,   B,    ldb,      N,  C,
                    ldc,  table, order, sums,  items,  keep,  cut_rows, lg, xcd_remap,
                    static_cast<hipStream_t>(stream)};
  const bool p32 = rowptr_bits == 32;
  if (dtype == FSP_F64)
    return p32 ? launch_ptr<double, double, int>(a, vec)
               : launch_ptr<double, double, int64_t>(a, vec);
  if (acc_f64)
    return p32 ? launch_ptr<float, double, int>(a, vec)
               : launch_ptr<float, double, int64_t>(a, vec);
  return p32 ? launch_ptr<float, float, int>(a, vec) : launch_ptr<float, float, int64_t>(a, vec);
}
