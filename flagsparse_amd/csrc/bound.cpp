// Calls with everything but the input, the output and the stream filled in.
//
// A prepared matrix is multiplied many times, and a small product is over in 4 us: converting
// its two dozen arguments from Python again for every call took longer than the launch.  A bound
// call holds them in a block of the caller's memory; fsp_run hands them, with the call's own
// three, to the same entry point, which checks them as ever.
#include <new>

#include "fsp_internal.hpp"

namespace {

constexpr uint64_t kMagic = 0x6673705f63616c6cULL;

enum Kind { kSpmvCsr, kSpmvSliced, kSpmmCsr, kSpmmSliced };

struct SpmvCsr {
  int dtype, acc_f64;
  const void* vals;
  const int32_t* cols;
  const void* rowptr;
  int rowptr_bits;
  int64_t n_rows, nnz;
  const int32_t* row_map;
  int64_t n_out;
  const int32_t* desc;
  const int64_t* ranges;
  int64_t n_desc, chunk;
  void* partials;
  const int32_t* groups;
  const int64_t* group_base;
  const int32_t* split_rows;
  int64_t n_groups;
  int xcd_remap;
};

struct SpmvSliced {
  int dtype, acc_f64;
  const void* vals;
  const int32_t* cols;
  const void* rowptr;
  int rowptr_bits;
  int64_t n_rows, nnz;
  int64_t* table;
  int table_built;
  void* sums;
  int cut_rows;
};

struct SpmmCsr {
  int dtype, acc_f64;
  const void* vals;
  const int32_t* cols;
  const void* rowptr;
  int rowptr_bits;
  int64_t n_rows, nnz, N;
  const int32_t* desc;
  int64_t n_desc, chunk;
  int lanes, vec;
  void* partials;
  const int32_t* groups;
  const int64_t* group_base;
  const int32_t* split_rows;
  int64_t n_groups;
  int xcd_remap;
};

struct SpmmSliced {
  int dtype, acc_f64;
  const void* vals;
  const int32_t* cols;
  const void* rowptr;
  int rowptr_bits;
  int64_t n_rows, nnz, N;
  const int64_t* table;
  const int32_t* order;
  int64_t items, keep;
  void* sums;
  int cut_rows, lanes, vec, xcd_remap;
};

struct Bound {
  uint64_t magic;
  int kind;
  union {
    SpmvCsr spmv;
    SpmvSliced spmv_sliced;
    SpmmCsr spmm;
    SpmmSliced spmm_sliced;
  };
};

Bound* bound_at(void* call, int kind) {
  if (!call || reinterpret_cast<uintptr_t>(call) % alignof(Bound)) return nullptr;
  Bound* b = ::new (call) Bound;
  b->magic = kMagic;
  b->kind = kind;
  return b;
}

int bad(const char* who) {
  return fsp::set_error(FSP_EINVAL, std::string(who) + ": call must be 8-byte aligned memory of "
                                                       "fsp_bound_bytes() bytes");
}

}  // namespace

extern "C" int64_t fsp_bound_bytes(void) { return sizeof(Bound); }

extern "C" int fsp_bind_spmv_csr(void* call, int dtype, int acc_f64, const void* vals,
                                 const int32_t* cols, const void* rowptr, int rowptr_bits,
                                 int64_t n_rows, int64_t nnz, const int32_t* row_map,
                                 int64_t n_out, const int32_t* desc, const int64_t* ranges,
                                 int64_t n_desc, int64_t chunk, void* partials,
                                 const int32_t* groups, const int64_t* group_base,
                                 const int32_t* split_rows, int64_t n_groups, int xcd_remap) {
  Bound* b = bound_at(call, kSpmvCsr);
  if (!b) return bad("fsp_bind_spmv_csr");
  b->spmv = {dtype, acc_f64, vals,  cols,     rowptr, rowptr_bits, n_rows,     nnz,        row_map, n_out,
             desc,  ranges,  n_desc, chunk, partials, groups, group_base, split_rows, n_groups, xcd_remap};
  return FSP_OK;
}

extern "C" int fsp_bind_spmv_sliced(void* call, int dtype, int acc_f64, const void* vals,
                                    const int32_t* cols, const void* rowptr, int rowptr_bits,
                                    int64_t n_rows, int64_t nnz, int64_t* table,
                                    int table_built, void* sums, int cut_rows) {
  Bound* b = bound_at(call, kSpmvSliced);
  if (!b) return bad("fsp_bind_spmv_sliced");
  b->spmv_sliced = {dtype,  acc_f64, vals,  cols,        rowptr, rowptr_bits,
                    n_rows, nnz,     table, table_built, sums,   cut_rows};
  return FSP_OK;
}

extern "C" int fsp_bind_spmm_csr(void* call, int dtype, int acc_f64, const void* vals,
                                 const int32_t* cols, const void* rowptr, int rowptr_bits,
                                 int64_t n_rows, int64_t nnz, int64_t N, const int32_t* desc,
                                 int64_t n_desc, int64_t chunk, int lanes_per_row, int vec,
                                 void* partials, const int32_t* groups,
                                 const int64_t* group_base, const int32_t* split_rows,
                                 int64_t n_groups, int xcd_remap) {
  Bound* b = bound_at(call, kSpmmCsr);
  if (!b) return bad("fsp_bind_spmm_csr");
  b->spmm = {dtype, acc_f64, vals,          cols, rowptr,   rowptr_bits, n_rows,     nnz,        N,        desc,
             n_desc, chunk,  lanes_per_row, vec,  partials, groups,      group_base, split_rows, n_groups, xcd_remap};
  return FSP_OK;
}

extern "C" int fsp_bind_spmm_sliced(void* call, int dtype, int acc_f64, const void* vals,
                                    const int32_t* cols, const void* rowptr, int rowptr_bits,
                                    int64_t n_rows, int64_t nnz, int64_t N,
                                    const int64_t* table, const int32_t* order, int64_t items,
                                    int64_t keep, void* sums, int cut_rows, int lanes_per_row,
                                    int vec, int xcd_remap) {
  Bound* b = bound_at(call, kSpmmSliced);
  if (!b) return bad("fsp_bind_spmm_sliced");
  b->spmm_sliced = {dtype, acc_f64, vals,  cols, rowptr, rowptr_bits,   n_rows, nnz,      N,
                    table, order,   items, keep, sums,   cut_rows, lanes_per_row, vec, xcd_remap};
  return FSP_OK;
}

extern "C" int fsp_run(const void* call, const void* in, void* out, void* stream) {
  const Bound* b = static_cast<const Bound*>(call);
  if (!b || b->magic != kMagic) return fsp::set_error(FSP_EINVAL, "fsp_run: not a bound call");
  switch (b->kind) {
    case kSpmvCsr: {
      const SpmvCsr& a = b->spmv;
      return fsp_spmv_csr(a.dtype, a.acc_f64, a.vals, a.cols, a.rowptr, a.rowptr_bits, a.n_rows,
                          a.nnz, in, out, a.row_map, a.n_out, a.desc, a.ranges, a.n_desc, a.chunk,
                          a.partials, a.groups, a.group_base, a.split_rows, a.n_groups,
                          a.xcd_remap, stream);
    }
    case kSpmvSliced: {
      const SpmvSliced& a = b->spmv_sliced;
      return fsp_spmv_sliced(a.dtype, a.acc_f64, a.vals, a.cols, a.rowptr, a.rowptr_bits,
                             a.n_rows, a.nnz, in, out, a.table, a.table_built, a.sums, a.cut_rows,
                             stream);
    }
    case kSpmmCsr: {
      const SpmmCsr& a = b->spmm;
      return fsp_spmm_csr(a.dtype, a.acc_f64, a.vals, a.cols, a.rowptr, a.rowptr_bits, a.n_rows,
                          a.nnz, in, a.N, a.N, out, a.N, a.desc, a.n_desc, a.chunk, a.lanes,
                          a.vec, a.partials, a.groups, a.group_base, a.split_rows, a.n_groups,
                          a.xcd_remap, stream);
    }
    default: {
      const SpmmSliced& a = b->spmm_sliced;
      return fsp_spmm_sliced(a.dtype, a.acc_f64, a.vals, a.cols, a.rowptr, a.rowptr_bits,
                             a.n_rows, a.nnz, in, a.N, a.N, out, a.N, a.table, a.order, a.items,
                             a.keep, a.sums, a.cut_rows, a.lanes, a.vec, a.xcd_remap, stream);
    }
  }
}
