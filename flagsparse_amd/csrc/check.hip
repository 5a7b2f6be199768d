// Structural checks of CSR and COO index arrays in one device pass, with their narrowing.
//
// A call on a matrix that was not prepared must know, before any kernel gathers through the
// arrays, that every index lies inside the matrix (CSR: that the row pointers start at 0, end at
// nnz and never decrease; COO: whether the rows are in order), and reads int32 copies of int64
// arrays.  As torch reductions, comparisons and casts those were about a dozen launches, each
// reading the arrays again.  Here one launch reads each array once, and every workgroup stores
// its result in pinned host memory, where the host waits for the words and reduces them: no
// second launch, no copy back, and no wait for the stream's completion signal.  (Measured on
// MI355X from launch to result, 16k entries: two launches, device copy and stream wait 20.8 us;
// result in pinned memory and stream wait 17.7; words watched 13.3; with the call from Python around
// it, two launches and a copy 26.3, one launch and watched words 16.0.)
//
// Reference behaviour replaced: the per-call checks of spmv_csr.py:379-436,
// spmm_csr.py:197-255, sddmm_csr.py:46-79 and spmm_coo.py:312-371.
//
// Bound: the index bytes at HBM rate, for small matrices the launch and the wait.  Measured on
// MI355X, 12.0M int64 columns and 1.0M int64 row pointers (104 MB read, 52 MB written): 28.5 us,
// 5.5 TB/s; torch's reductions and casts took 130 us in 40 launches.
#include <chrono>
#include <climits>

#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

typedef int64_t i64x2 __attribute__((ext_vector_type(2)));

// Few, large workgroups: every one stores into host memory, across the bus (1.65M COO entries:
// 806 workgroups of 256 threads with five stores each took 30 us longer than a second launch).
constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int64_t kStep = 4 * kThreads;  // elements a workgroup takes in one step
constexpr int kCsrWords = 2;  // per workgroup: {min, ~max} of columns or {decreases, longest}
constexpr int kRowWords = 4;  // the same, and from row pointers {uneven rows, entries in cut rows}
constexpr int kCooWords = 5;  // {min, ~max} of rows, {min, ~max} of columns, decreases
// What a word holds until its workgroup has stored it.
constexpr int64_t kPending = LLONG_MIN + 0x5bd1e995;

__device__ __forceinline__ int64_t wave_min_i64(int64_t v) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t o = __shfl_xor(v, off, kWave);
    v = o < v ? o : v;
  }
  return v;
}

__device__ __forceinline__ int64_t wave_add_i64(int64_t v) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Minimum (or, with ADD, sum) over the workgroup, in every thread; s_w holds a word per wave.
template <bool ADD>
__device__ __forceinline__ int64_t block_reduce(int64_t v, int64_t* s_w) {
  v = ADD ? wave_add_i64(v) : wave_min_i64(v);
  __syncthreads();  // s_w may still be read by a previous call
  if ((threadIdx.x & (kWave - 1)) == 0) s_w[threadIdx.x / kWave] = v;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const int64_t o = s_w[w];
    if (w == 0) v = o;
    else if (ADD) v += o;
    else v = o < v ? o : v;
  }
  return v;
}

// Four elements at p (the first of a quad); vec: p is 16-byte aligned.
template <typename I>
__device__ __forceinline__ void load4(const I* p, bool vec, I (&v)[4]) {
  if (vec) {
    if constexpr (sizeof(I) == 4) {
      const i32x4 q = *reinterpret_cast<const i32x4*>(p);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
      const i64x2 a = reinterpret_cast<const i64x2*>(p)[0];
      const i64x2 b = reinterpret_cast<const i64x2*>(p)[1];
      v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = p[j];
  }
}

template <typename I>
__device__ __forceinline__ void store4(int32_t* out, const I (&v)[4]) {
  i32x4 o;
  o.x = (int)v[0]; o.y = (int)v[1]; o.z = (int)v[2]; o.w = (int)v[3];
  *reinterpret_cast<i32x4*>(out) = o;
}

template <typename I>
struct Bounds {
  I mn = sizeof(I) == 4 ? (I)INT_MAX : (I)LLONG_MAX;
  I mx = sizeof(I) == 4 ? (I)INT_MIN : (I)LLONG_MIN;
  __device__ __forceinline__ void add(I v) {
    mn = v < mn ? v : mn;
    mx = v > mx ? v : mx;
  }
  // ~x reverses the order without overflow: both ends reduce as minima.
  __device__ __forceinline__ int64_t low() const { return (int64_t)mn; }
  __device__ __forceinline__ int64_t high() const { return ~(int64_t)mx; }
};

__device__ __forceinline__ void publish(int64_t* host, int64_t v) {
  __hip_atomic_store(host, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What else is counted of the rows (COUNT): those of more than `uneven` and at most `block` entries,
// and the entries of those of more than `chunk`.
struct RowClasses {
  int64_t uneven, block, chunk;
};

// host: [0] = ptr[0], [1] = ptr[n_rows], then kCsrWords or, with COUNT, kRowWords per workgroup.
template <typename I, typename P, bool COUNT>
__global__ __launch_bounds__(kThreads) void csr_check_kernel(
    const I* __restrict__ idx, int64_t nnz, const P* __restrict__ ptr, int64_t n_rows,
    int32_t* __restrict__ idx32, void* __restrict__ ptr_out, int ptr_out_bits, int idx_vec,
    int idx_blocks, RowClasses rows, int64_t* host) {
  __shared__ int64_t s_w[kWaves];
  const int tid = threadIdx.x;
  int64_t a, b, uneven = 0, cut = 0;
  if ((int)blockIdx.x < idx_blocks) {
    Bounds<I> c;
    const int64_t stride = (int64_t)idx_blocks * kStep;
    for (int64_t i = (int64_t)blockIdx.x * kStep + 4 * tid; i < nnz; i += stride) {
      if (i + 4 <= nnz) {
        I v[4];
        load4<I>(idx + i, idx_vec != 0, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) c.add(v[j]);
        if (idx32) store4<I>(idx32 + i, v);  // 16-byte aligned; i is a multiple of 4
      } else {
        for (int64_t j = i; j < nnz; ++j) {
          c.add(idx[j]);
          if (idx32) idx32[j] = (int)idx[j];
        }
      }
    }
    a = block_reduce<false>(c.low(), s_w);
    b = block_reduce<false>(c.high(), s_w);
  } else {
    const int64_t blk = (int64_t)blockIdx.x - idx_blocks;
    const int64_t stride = (int64_t)(gridDim.x - idx_blocks) * kThreads;
    int64_t dec = 0, longest = 0;
    // pointer i (0 .. n_rows) is copied by its thread, which also looks at row i
    for (int64_t i = blk * kThreads + tid; i <= n_rows; i += stride) {
      const int64_t p = (int64_t)ptr[i];
      if (ptr_out) {
        if (ptr_out_bits == 32) static_cast<int32_t*>(ptr_out)[i] = (int32_t)p;
        else static_cast<int64_t*>(ptr_out)[i] = p;
      }
      if (i == 0) publish(host, p);
      if (i == n_rows) publish(host + 1, p);
      if (i < n_rows) {
        const int64_t q = (int64_t)ptr[i + 1];
        const int64_t len = (int64_t)((uint64_t)q - (uint64_t)p);
        dec += q < p ? 1 : 0;
        longest = len > longest ? len : longest;
        if constexpr (COUNT) {
          uneven += len > rows.uneven && len <= rows.block ? 1 : 0;
          cut += len > rows.chunk ? len : 0;
        }
      }
    }
    if constexpr (!COUNT) a = block_reduce<true>(dec, s_w);
    b = block_reduce<false>(~longest, s_w);
    if constexpr (COUNT) {  // the three sums behind one barrier
      __shared__ int64_t s_sum[3][kWaves];
      const int64_t d = wave_add_i64(dec), u = wave_add_i64(uneven), c = wave_add_i64(cut);
      if ((tid & (kWave - 1)) == 0) {
        s_sum[0][tid / kWave] = d;
        s_sum[1][tid / kWave] = u;
        s_sum[2][tid / kWave] = c;
      }
      __syncthreads();
      a = uneven = cut = 0;
      for (int w = 0; w < kWaves; ++w) {
        a += s_sum[0][w];
        uneven += s_sum[1][w];
        cut += s_sum[2][w];
      }
    }
  }
  constexpr int kWords = COUNT ? kRowWords : kCsrWords;
  if (tid < kWords)  // one store
    publish(host + 2 + (int64_t)blockIdx.x * kWords + tid,
            tid == 0 ? a : !COUNT || tid == 1 ? b : tid == 2 ? uneven : cut);
}

// host: kCooWords per workgroup.  row32 / col32: NULL, or the narrowed arrays.
template <typename R, typename C>
__global__ __launch_bounds__(kThreads) void coo_check_kernel(const R* __restrict__ row,
                                                           const C* __restrict__ col,
                                                           int64_t nnz, int32_t* __restrict__ row32,
                                                           int32_t* __restrict__ col32, int row_vec,
                                                           int col_vec, int64_t* host) {
  __shared__ int64_t s_w[kWaves];
  Bounds<R> r;
  Bounds<C> c;
  int64_t dec = 0;
  const int64_t stride = (int64_t)gridDim.x * kStep;
  for (int64_t i = (int64_t)blockIdx.x * kStep + 4 * threadIdx.x; i < nnz; i += stride) {
    const R before = i > 0 ? row[i - 1] : row[0];
    if (i + 4 <= nnz) {
      R u[4];
      C v[4];
      load4<R>(row + i, row_vec != 0, u);
      load4<C>(col + i, col_vec != 0, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        r.add(u[j]);
        c.add(v[j]);
      }
      dec += (u[0] < before) + (u[1] < u[0]) + (u[2] < u[1]) + (u[3] < u[2]);
      if (row32) store4<R>(row32 + i, u);
      if (col32) store4<C>(col32 + i, v);
    } else {
      R prev = before;
      for (int64_t j = i; j < nnz; ++j) {
        r.add(row[j]);
        c.add(col[j]);
        dec += row[j] < prev ? 1 : 0;
        prev = row[j];
        if (row32) row32[j] = (int)row[j];
        if (col32) col32[j] = (int)col[j];
      }
    }
  }
  int64_t w[kCooWords];
  w[0] = block_reduce<false>(r.low(), s_w);
  w[1] = block_reduce<false>(r.high(), s_w);
  w[2] = block_reduce<false>(c.low(), s_w);
  w[3] = block_reduce<false>(c.high(), s_w);
  w[4] = block_reduce<true>(dec, s_w);
  if (threadIdx.x < kCooWords) {  // one store
    int64_t mine = w[0];
#pragma unroll
    for (int k = 1; k < kCooWords; ++k) mine = threadIdx.x == k ? w[k] : mine;
    publish(host + (int64_t)blockIdx.x * kCooWords + threadIdx.x, mine);
  }
}

int64_t blocks_for(int64_t n, int64_t per, int64_t cap) {
  const int64_t b = (n + per - 1) / per;
  return b < 1 ? int64_t(1) : b > cap ? cap : b;
}

// Waits until the n words at host are stored.  A word is a result by itself, so seeing it is
// enough; after kSpin without one (work queued before the check, a word that happens to be
// kPending, host memory the device does not write through to) the stream's completion decides.
int wait_words(const int64_t* host, int64_t n, hipStream_t st) {
  constexpr auto kSpin = std::chrono::microseconds(200);
  const volatile int64_t* p = host;
  const auto start = std::chrono::steady_clock::now();
  for (int64_t i = 0, turns = 0; i < n; ++i) {
    while (p[i] == kPending) {
      if ((++turns & 63) == 0 && std::chrono::steady_clock::now() - start > kSpin)
        return check_hip(hipStreamSynchronize(st), "index check");
    }
  }
  return FSP_OK;
}

template <typename I, typename P, bool COUNT>
int run_csr_check(const void* idx, int64_t nnz, const void* ptr, int64_t n_rows, int32_t* idx32,
                  void* ptr_out, int ptr_out_bits, const RowClasses& rows, int64_t* pinned,
                  int64_t* out, hipStream_t st) {
  const int64_t ib = nnz > 0 ? blocks_for(nnz, kStep, kCheckBlocks) : 0;
  const int64_t pb = blocks_for(n_rows + 1, 2 * kThreads, kCheckBlocks / 4);
  constexpr int kWords = COUNT ? kRowWords : kCsrWords;
  const int64_t n = 2 + (ib + pb) * kWords;
  for (int64_t i = 0; i < n; ++i) pinned[i] = kPending;
  const int vec = reinterpret_cast<uintptr_t>(idx) % 16 == 0;
  hipLaunchKernelGGL((csr_check_kernel<I, P, COUNT>), dim3((unsigned)(ib + pb)), dim3(kThreads), 0, st,
                     static_cast<const I*>(idx), nnz, static_cast<const P*>(ptr), n_rows, idx32,
                     ptr_out, ptr_out_bits, vec, (int)ib, rows, pinned);
  int rc = check_hip(hipGetLastError(), "csr_check_kernel launch");
  if (!rc) rc = wait_words(pinned, n, st);
  if (rc) return rc;
  int64_t mn = LLONG_MAX, nmx = LLONG_MAX, dec = 0, nlong = ~int64_t(0), uneven = 0, cut = 0;
  for (int64_t b = 0; b < ib + pb; ++b) {
    const int64_t* w = pinned + 2 + b * kWords;
    const int64_t u = w[0], v = w[1];
    if constexpr (COUNT) {
      uneven += w[2];
      cut += w[3];
    }
    if (b < ib) {
      mn = u < mn ? u : mn;
      nmx = v < nmx ? v : nmx;
    } else {
      dec += u;
      nlong = v < nlong ? v : nlong;
    }
  }
  out[0] = pinned[0];
  out[1] = pinned[1];
  out[2] = dec;
  out[3] = ~nlong;
  out[4] = mn;
  out[5] = ~nmx;
  if constexpr (COUNT) {
    out[6] = uneven;
    out[7] = cut;
  }
  return FSP_OK;
}

template <typename R, typename C>
int run_coo_check(const void* row, const void* col, int64_t nnz, int32_t* row32, int32_t* col32,
                  int64_t* pinned, int64_t* out, hipStream_t st) {
  const int64_t blocks = blocks_for(nnz, kStep, kCheckBlocks);
  const int64_t n = blocks * kCooWords;
  for (int64_t i = 0; i < n; ++i) pinned[i] = kPending;
  hipLaunchKernelGGL((coo_check_kernel<R, C>), dim3((unsigned)blocks), dim3(kThreads), 0, st,
                     static_cast<const R*>(row), static_cast<const C*>(col), nnz, row32, col32,
                     (int)(reinterpret_cast<uintptr_t>(row) % 16 == 0),
                     (int)(reinterpret_cast<uintptr_t>(col) % 16 == 0), pinned);
  int rc = check_hip(hipGetLastError(), "coo_check_kernel launch");
  if (!rc) rc = wait_words(pinned, n, st);
  if (rc) return rc;
  int64_t w[kCooWords] = {LLONG_MAX, LLONG_MAX, LLONG_MAX, LLONG_MAX, 0};
  for (int64_t b = 0; b < blocks; ++b) {
    for (int k = 0; k < 4; ++k) {
      const int64_t v = pinned[b * kCooWords + k];
      w[k] = v < w[k] ? v : w[k];
    }
    w[4] += pinned[b * kCooWords + 4];
  }
  out[0] = w[0];
  out[1] = ~w[1];
  out[2] = w[2];
  out[3] = ~w[3];
  out[4] = w[4];
  return FSP_OK;
}

}  // namespace
}  // namespace fsp

using namespace fsp;

extern "C" int64_t fsp_check_pinned_len(void) {
  const int64_t csr = 2 + 2 * kCheckBlocks * kRowWords, coo = kCheckBlocks * kCooWords;
  return csr > coo ? csr : coo;
}

namespace {

template <bool COUNT>
int csr_check(const void* indices, int idx_bits, int64_t nnz, const void* indptr, int ptr_bits,
              int64_t n_rows, int32_t* idx32, void* ptr_out, int ptr_out_bits,
              const RowClasses& rows, int64_t* pinned, int64_t* out, void* stream) {
  if ((idx_bits != 32 && idx_bits != 64) || (ptr_bits != 32 && ptr_bits != 64) ||
      (ptr_out && ptr_out_bits != 32 && ptr_out_bits != 64))
    return set_error(FSP_EINVAL, "fsp_csr_check: index widths must be 32 or 64");
  if (nnz < 0 || n_rows < 0) return set_error(FSP_EINVAL, "fsp_csr_check: negative size");
  if (!indptr || !pinned || !out || (nnz > 0 && !indices))
    return set_error(FSP_EINVAL, "fsp_csr_check: null pointer");
  if (reinterpret_cast<uintptr_t>(idx32) % 16)
    return set_error(FSP_EINVAL, "fsp_csr_check: idx32 must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define FSP_CHECK_ARGS indices, nnz, indptr, n_rows, idx32, ptr_out, ptr_out_bits, rows, pinned, out, st
  if (idx_bits == 32)
    return ptr_bits == 32 ? run_csr_check<int32_t, int32_t, COUNT>(FSP_CHECK_ARGS)
                          : run_csr_check<int32_t, int64_t, COUNT>(FSP_CHECK_ARGS);
  return ptr_bits == 32 ? run_csr_check<int64_t, int32_t, COUNT>(FSP_CHECK_ARGS)
                        : run_csr_check<int64_t, int64_t, COUNT>(FSP_CHECK_ARGS);
#undef FSP_CHECK_ARGS
}

}  // namespace

extern "C" int fsp_csr_check(const void* indices, int idx_bits, int64_t nnz, const void* indptr,
                             int ptr_bits, int64_t n_rows, int32_t* idx32, void* ptr_out,
                             int ptr_out_bits, int64_t* pinned, int64_t* out, void* stream) {
  return csr_check<false>(indices, idx_bits, nnz, indptr, ptr_bits, n_rows, idx32, ptr_out,
                          ptr_out_bits, RowClasses{0, 0, 0}, pinned, out, stream);
}

extern "C" int fsp_csr_check_rows(const void* indices, int idx_bits, int64_t nnz,
                                  const void* indptr, int ptr_bits, int64_t n_rows,
                                  int32_t* idx32, void* ptr_out, int ptr_out_bits, int64_t uneven,
                                  int64_t block, int64_t chunk, int64_t* pinned, int64_t* out,
                                  void* stream) {
  return csr_check<true>(indices, idx_bits, nnz, indptr, ptr_bits, n_rows, idx32, ptr_out,
                         ptr_out_bits, RowClasses{uneven, block, chunk}, pinned, out, stream);
}

extern "C" int fsp_coo_check(const void* rows, int row_bits, const void* cols, int col_bits,
                             int64_t nnz, int32_t* row32, int32_t* col32, int64_t* pinned,
                             int64_t* out, void* stream) {
  if ((row_bits != 32 && row_bits != 64) || (col_bits != 32 && col_bits != 64))
    return set_error(FSP_EINVAL, "fsp_coo_check: index widths must be 32 or 64");
  if (nnz < 1) return set_error(FSP_EINVAL, "fsp_coo_check: nnz must be >= 1");
  if (!rows || !cols || !pinned || !out)
    return set_error(FSP_EINVAL, "fsp_coo_check: null pointer");
  if (reinterpret_cast<uintptr_t>(row32) % 16 || reinterpret_cast<uintptr_t>(col32) % 16)
    return set_error(FSP_EINVAL, "fsp_coo_check: row32 and col32 must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (row_bits == 32 && col_bits == 32)
    return run_coo_check<int32_t, int32_t>(rows, cols, nnz, row32, col32, pinned, out, st);
  if (row_bits == 32)
    return run_coo_check<int32_t, int64_t>(rows, cols, nnz, row32, col32, pinned, out, st);
  if (col_bits == 32)
    return run_coo_check<int64_t, int32_t>(rows, cols, nnz, row32, col32, pinned, out, st);
  return run_coo_check<int64_t, int64_t>(rows, cols, nnz, row32, col32, pinned, out, st);
}
