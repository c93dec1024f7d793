// Rows whose width or alignment fits no 16-byte layout (fp32 at any width,
// bf16 at even widths): what the kernels that hold such a row in one
// workgroup's registers share.
//
// A row starts at any 4-byte address.  dwordx4 buffer loads and stores need no
// more than that, and a raw buffer's range check works per dword: with
// num_records the row's bytes, the row's last vector reads zeros past the end
// and its stores there are dropped, so a ragged row runs the same
// straight-line code as an aligned one.  Only identities other than zero need
// a mask (keep4).
//
// The workgroups are persistent: as many as the device holds at once, each
// taking rows blockIdx, blockIdx + grid, ..., and as a row's outputs leave its
// registers the next row's loads are issued into them, so loads and stores
// overlap without a second set of registers.
#pragma once

#include "api_internal.hpp"
#include "common.hpp"

namespace credit {
namespace rows {

template <class T>
__device__ __forceinline__ buffer_rsrc_t row_rsrc(const T* base, int row, int rows, int cols) {
  return make_rsrc(base + static_cast<size_t>(row < rows ? row : 0) * cols,
                   row < rows ? static_cast<uint32_t>(cols * sizeof(T)) : 0u);
}
__device__ __forceinline__ f32x4 row_load(buffer_rsrc_t r, uint32_t offset) {
  return __builtin_bit_cast(f32x4, buffer_load_nt(r, offset));
}
__device__ __forceinline__ void row_store(buffer_rsrc_t r, uint32_t offset, f32x4 v) {
  buffer_store_nt(r, offset, __builtin_bit_cast(u32x4, v));
}

// v with `fill` in the elements past the row's end; left: the row's elements
// from this vector's first one on (may be negative).
__device__ __forceinline__ f32x4 keep4(f32x4 v, int left, float fill) {
  return f32x4{left > 0 ? v.x : fill, left > 1 ? v.y : fill, left > 2 ? v.z : fill,
               left > 3 ? v.w : fill};
}

// Block reductions on an LDS-only barrier (loads and stores in flight stay
// so).  A slot array is rewritten only after two later barriers, so no
// trailing one is needed.
template <int NW>
__device__ __forceinline__ float block_max(float v, float* slots) {
  v = wave_reduce(v, MaxOp{});
  if ((threadIdx.x & (kWave - 1)) == 0) slots[threadIdx.x / kWave] = v;
  lds_barrier();
  float r = slots[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) r = fmax_nan(r, slots[w]);
  return r;
}
template <int NW>
__device__ __forceinline__ double block_sum(double v, double* slots) {
  v = wave_reduce_sum_f64(v);
  if ((threadIdx.x & (kWave - 1)) == 0) slots[threadIdx.x / kWave] = v;
  lds_barrier();
  double r = slots[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) r += slots[w];
  return r;
}

template <int NW>
__device__ __forceinline__ void block_sum2(double& a, double& b, double (*slots)[NW]) {
  a = wave_reduce_sum_f64(a);
  b = wave_reduce_sum_f64(b);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    slots[0][threadIdx.x / kWave] = a;
    slots[1][threadIdx.x / kWave] = b;
  }
  lds_barrier();
  a = slots[0][0];
  b = slots[1][0];
#pragma unroll
  for (int w = 1; w < NW; ++w) {
    a += slots[0][w];
    b += slots[1][w];
  }
}

// fp32 vectors at 4-byte addresses, for the kernels that stream a row wider
// than one workgroup's registers (global loads: a row may pass 4 GiB).
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f32x4 stream_load(const float* row, int vec) {
  return __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4*>(row) + vec);
}
__device__ __forceinline__ void stream_store(float* row, int vec, f32x4 v) {
  __builtin_nontemporal_store(static_cast<f32x4_a4>(v), reinterpret_cast<f32x4_a4*>(row) + vec);
}
// Few rows: one workgroup streams a whole row, so a wide one.
inline unsigned stream_threads(int64_t rows) { return rows < 1024 ? 1024 : 256; }

template <class Fn>
struct RowsPick {
  Fn fn;
  int threads;
  int64_t capacity;  // elements
};

// The narrowest entry that holds `cols`; nullptr: none.
template <class Fn, int N>
const RowsPick<Fn>* rows_pick(const RowsPick<Fn> (&table)[N], int64_t cols) {
  for (const RowsPick<Fn>& p : table)
    if (cols <= p.capacity) return &p;
  return nullptr;
}

// The persistent grid of a pick over `rows` rows.
template <class Fn>
int rows_grid(const RowsPick<Fn>& pick, int64_t rows, unsigned* grid) {
  if (rows <= 256) {  // at most one row per CU: no query needed
    *grid = static_cast<unsigned>(rows);
    return CREDIT_OK;
  }
  int64_t fit = 0;
  CREDIT_TRY(resident_workgroups(reinterpret_cast<const void*>(pick.fn), pick.threads, 0, &fit));
  *grid = static_cast<unsigned>(rows < fit ? rows : fit);
  return CREDIT_OK;
}

}  // namespace rows
}  // namespace credit
