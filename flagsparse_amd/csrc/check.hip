// Structural checks of a CSR matrix in one device pass, with the narrowing of its index arrays.
//
// A call on a matrix that was not prepared must know, before any kernel gathers through the
// arrays, that the row pointers start at 0, end at nnz and never decrease and that every
// column lies inside the matrix; it also needs the longest row, and int32 copies of int64
// arrays.  As torch reductions, comparisons and casts those were about a dozen launches, each
// reading the arrays again.  Here workgroups [0, idx_blocks) read the columns once (minimum,
// maximum, int32 copy) and the others read the row pointers once (decreases, longest row,
// narrowed copy); a second, one-workgroup launch reduces the partials in a fixed order and
// adds the first and last row pointer.
//
// Reference behaviour replaced: the per-call checks of spmv_csr.py:379-436,
// spmm_csr.py:197-255 and sddmm_csr.py:46-79.
//
// Bound: the index bytes at HBM rate, for small matrices the two launches.  Measured on MI355X,
// 12.0M int64 columns and 1.0M int64 row pointers (104 MB read, 52 MB written): 24 us, 6.5 TB/s,
// and 5.7 us for the second launch; torch's reductions and casts took 130 us in 40 launches.
#include <climits>

#include "fsp_device.hpp"
#include "fsp_internal.hpp"

namespace fsp {
namespace {

typedef int64_t i64x2 __attribute__((ext_vector_type(2)));
constexpr int kPartials = 2;  // per workgroup: {min, max} of the columns or {decreases, longest}
// Elements a workgroup takes in one step (4 per thread); a workgroup of the first launch gets
// at least kMinSteps steps, so that small arrays do not pay for many workgroups' reductions.
constexpr int64_t kStep = 4 * kBlock;
constexpr int64_t kMinSteps = 2;

__device__ __forceinline__ int64_t wave_min_i64(int64_t v) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t o = __shfl_xor(v, off, kWave);
    v = o < v ? o : v;
  }
  return v;
}

__device__ __forceinline__ int64_t wave_max_i64(int64_t v) { return -wave_min_i64(-v); }

__device__ __forceinline__ int64_t wave_add_i64(int64_t v) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Four elements at p (base element of a quad); vec: p is 16-byte aligned.
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

template <typename I, typename P>
__global__ __launch_bounds__(kBlock) void csr_check_kernel(
    const I* __restrict__ idx, int64_t nnz, const P* __restrict__ ptr, int64_t n_rows,
    int32_t* __restrict__ idx32, void* __restrict__ ptr_out, int ptr_out_bits, int idx_vec,
    int idx_blocks, int64_t* __restrict__ partial) {
  __shared__ int64_t s_a[kWavesPerBlock], s_b[kWavesPerBlock];
  const int tid = threadIdx.x;
  int64_t a, b;  // the workgroup's pair of partials
  const bool columns = (int)blockIdx.x < idx_blocks;
  if (columns) {
    I mn = sizeof(I) == 4 ? (I)INT_MAX : (I)LLONG_MAX;
    I mx = sizeof(I) == 4 ? (I)INT_MIN : (I)LLONG_MIN;
    const int64_t stride = (int64_t)idx_blocks * kStep;
    for (int64_t i = (int64_t)blockIdx.x * kStep + 4 * tid; i < nnz; i += stride) {
      if (i + 4 <= nnz) {
        I v[4];
        load4<I>(idx + i, idx_vec != 0, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          mn = v[j] < mn ? v[j] : mn;
          mx = v[j] > mx ? v[j] : mx;
        }
        if (idx32) {  // a fresh, 16-byte aligned array; i is a multiple of 4
          i32x4 o;
          o.x = (int)v[0]; o.y = (int)v[1]; o.z = (int)v[2]; o.w = (int)v[3];
          *reinterpret_cast<i32x4*>(idx32 + i) = o;
        }
      } else {
        for (int64_t j = i; j < nnz; ++j) {
          const I v = idx[j];
          mn = v < mn ? v : mn;
          mx = v > mx ? v : mx;
          if (idx32) idx32[j] = (int)v;
        }
      }
    }
    a = wave_min_i64((int64_t)mn);
    b = wave_min_i64(~(int64_t)mx);  // ~x is order-reversing and has no overflow
  } else {
    const int64_t blk = (int64_t)blockIdx.x - idx_blocks;
    const int64_t stride = (int64_t)(gridDim.x - idx_blocks) * kBlock;
    int64_t dec = 0, longest = 0;
    // pointer i (0 .. n_rows) is copied by its thread, which also looks at row i
    for (int64_t i = blk * kBlock + tid; i <= n_rows; i += stride) {
      const int64_t p = (int64_t)ptr[i];
      if (ptr_out) {
        if (ptr_out_bits == 32) static_cast<int32_t*>(ptr_out)[i] = (int32_t)p;
        else static_cast<int64_t*>(ptr_out)[i] = p;
      }
      if (i < n_rows) {
        const int64_t q = (int64_t)ptr[i + 1];
        const int64_t len = (int64_t)((uint64_t)q - (uint64_t)p);
        dec += q < p ? 1 : 0;
        longest = len > longest ? len : longest;
      }
    }
    a = wave_add_i64(dec);
    b = wave_max_i64(longest);
  }
  if ((tid & (kWave - 1)) == 0) {
    s_a[tid / kWave] = a;
    s_b[tid / kWave] = b;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kWavesPerBlock; ++w) {
      if (columns) {
        a = s_a[w] < a ? s_a[w] : a;
        b = s_b[w] < b ? s_b[w] : b;
      } else {
        a += s_a[w];
        b = s_b[w] > b ? s_b[w] : b;
      }
    }
    partial[(int64_t)blockIdx.x * kPartials] = a;
    partial[(int64_t)blockIdx.x * kPartials + 1] = b;
  }
}

template <typename P>
__global__ __launch_bounds__(kBlock) void csr_check_final_kernel(
    const int64_t* __restrict__ partial, int idx_blocks, int all_blocks,
    const P* __restrict__ ptr, int64_t n_rows, int64_t* __restrict__ out) {
  __shared__ int64_t s[4][kWavesPerBlock];
  const int tid = threadIdx.x;
  int64_t mn = LLONG_MAX, nmx = LLONG_MAX, dec = 0, longest = 0;
  for (int b = tid; b < all_blocks; b += kBlock) {
    const int64_t u = partial[(int64_t)b * kPartials], v = partial[(int64_t)b * kPartials + 1];
    if (b < idx_blocks) {
      mn = u < mn ? u : mn;
      nmx = v < nmx ? v : nmx;
    } else {
      dec += u;
      longest = v > longest ? v : longest;
    }
  }
  mn = wave_min_i64(mn);
  nmx = wave_min_i64(nmx);
  dec = wave_add_i64(dec);
  longest = wave_max_i64(longest);
  if ((tid & (kWave - 1)) == 0) {
    const int w = tid / kWave;
    s[0][w] = mn; s[1][w] = nmx; s[2][w] = dec; s[3][w] = longest;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kWavesPerBlock; ++w) {
      mn = s[0][w] < mn ? s[0][w] : mn;
      nmx = s[1][w] < nmx ? s[1][w] : nmx;
      dec += s[2][w];
      longest = s[3][w] > longest ? s[3][w] : longest;
    }
    out[0] = (int64_t)ptr[0];
    out[1] = (int64_t)ptr[n_rows];
    out[2] = dec;
    out[3] = longest;
    out[4] = mn;
    out[5] = ~nmx;
  }
}

template <typename I, typename P>
int launch_check(const void* idx, int64_t nnz, const void* ptr, int64_t n_rows, int32_t* idx32,
                 void* ptr_out, int ptr_out_bits, int64_t* partial, int64_t* out,
                 hipStream_t st) {
  auto blocks_for = [](int64_t n, int64_t per, int64_t cap) {
    int64_t b = (n + per - 1) / per;
    return b < 1 ? int64_t(1) : b > cap ? cap : b;
  };
  const int64_t ib = nnz > 0 ? blocks_for(nnz, kMinSteps * kStep, kCsrCheckBlocks / 2) : 0;
  const int64_t pb = blocks_for(n_rows + 1, kMinSteps * kBlock, kCsrCheckBlocks / 2);
  const int vec = reinterpret_cast<uintptr_t>(idx) % 16 == 0;
  hipLaunchKernelGGL((csr_check_kernel<I, P>), dim3((unsigned)(ib + pb)), dim3(kBlock), 0, st,
                     static_cast<const I*>(idx), nnz, static_cast<const P*>(ptr), n_rows, idx32,
                     ptr_out, ptr_out_bits, vec, (int)ib, partial);
  int rc = check_hip(hipGetLastError(), "csr_check_kernel launch");
  if (rc) return rc;
  hipLaunchKernelGGL((csr_check_final_kernel<P>), dim3(1), dim3(kBlock), 0, st, partial, (int)ib,
                     (int)(ib + pb), static_cast<const P*>(ptr), n_rows, out);
  return check_hip(hipGetLastError(), "csr_check_final_kernel launch");
}

}  // namespace
}  // namespace fsp

using namespace fsp;

extern "C" int64_t fsp_csr_check_partial_len(void) { return kCsrCheckBlocks * kPartials; }

extern "C" int fsp_csr_check(const void* indices, int idx_bits, int64_t nnz, const void* indptr,
                             int ptr_bits, int64_t n_rows, int32_t* idx32, void* ptr_out,
                             int ptr_out_bits, int64_t* partial, int64_t* out, void* stream) {
  if ((idx_bits != 32 && idx_bits != 64) || (ptr_bits != 32 && ptr_bits != 64) ||
      (ptr_out && ptr_out_bits != 32 && ptr_out_bits != 64))
    return set_error(FSP_EINVAL, "fsp_csr_check: index widths must be 32 or 64");
  if (nnz < 0 || n_rows < 0) return set_error(FSP_EINVAL, "fsp_csr_check: negative size");
  if (!indptr || !partial || !out || (nnz > 0 && !indices))
    return set_error(FSP_EINVAL, "fsp_csr_check: null pointer");
  if (reinterpret_cast<uintptr_t>(idx32) % 16)
    return set_error(FSP_EINVAL, "fsp_csr_check: idx32 must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define FSP_CHECK_ARGS indices, nnz, indptr, n_rows, idx32, ptr_out, ptr_out_bits, partial, out, st
  if (idx_bits == 32)
    return ptr_bits == 32 ? launch_check<int32_t, int32_t>(FSP_CHECK_ARGS)
                          : launch_check<int32_t, int64_t>(FSP_CHECK_ARGS);
  return ptr_bits == 32 ? launch_check<int64_t, int32_t>(FSP_CHECK_ARGS)
                        : launch_check<int64_t, int64_t>(FSP_CHECK_ARGS);
#undef FSP_CHECK_ARGS
}
