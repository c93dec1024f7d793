// Rows whose width or alignment fits no 16-byte layout: what the kernels that
// hold such a row in one workgroup's registers share.
//
// An fp32 row, or a bf16 row of even width, starts at any 4-byte address (bf16
// rows of odd width: HalfRow below).  dwordx4 buffer loads and stores need no
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

#include <type_traits>

#include "api_internal.hpp"
#include "common.hpp"
#include "row_rules.hpp"

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

// A bf16 row of a tensor at a 4-byte address.  ODD (odd widths): every other
// row starts in the upper half of a dword.  It is then read from the dword's
// start, one dword further, and shifted into place; on the rows that start on
// a dword the last element shares its dword with the next row and travels by
// itself.  No access leaves the row's own elements but the half dword before
// an odd row's start, the previous row's last element.
struct HalfRow {
  buffer_rsrc_t dwords;  // the whole dwords from the row's first (half) dword on
  buffer_rsrc_t halves;  // the same to the row's last byte (ODD stores)
  uint32_t shift;        // 16 on an odd row, else 0
  uint32_t last;         // the row's last element (ODD loads)
};
// `n` elements (0: none) from element `at` on; more: the row goes on behind
// them (n a multiple of 8), so that an odd start's last dword, half of it the
// next element's, may be read whole.
template <bool ODD, bool LOAD>
__device__ __forceinline__ HalfRow half_span(const uint16_t* base, size_t at, uint32_t n,
                                             bool more) {
  const uint32_t odd = ODD ? static_cast<uint32_t>(at) & 1u : 0u;
  const uint32_t bytes = n > 0 ? (n + odd) * 2u : 0u;
  HalfRow r;
  r.dwords = make_rsrc(base + at - odd, (bytes + (ODD && more ? 2u : 0u)) & ~3u);
  r.halves = make_rsrc(base + at - odd, bytes);
  r.shift = odd * 16u;
  r.last = ODD && LOAD && n > 0 ? base[at + n - 1] : 0u;
  return r;
}
template <bool ODD, bool LOAD>
__device__ __forceinline__ HalfRow half_row(const uint16_t* base, int row, int rows, int cols) {
  const bool live = row < rows;
  return half_span<ODD, LOAD>(base, static_cast<size_t>(live ? row : 0) * cols,
                              live ? static_cast<uint32_t>(cols) : 0u, false);
}
// Elements 8 i .. 8 i + 7 of the row, off = 16 i, left = cols - 8 i; zeros past
// the row's end.
template <bool ODD, bool NT = true>
__device__ __forceinline__ u32x4 half_load(const HalfRow& r, uint32_t off, int left) {
  u32x4 v = NT ? buffer_load_nt(r.dwords, off) : buffer_load(r.dwords, off);
  if constexpr (ODD) {
    const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(r.dwords, off + 16u, 0, 0);
    v = u32x4{__builtin_amdgcn_alignbit(v.y, v.x, r.shift),
              __builtin_amdgcn_alignbit(v.z, v.y, r.shift),
              __builtin_amdgcn_alignbit(v.w, v.z, r.shift),
              __builtin_amdgcn_alignbit(w, v.w, r.shift)};
    // An odd width's last element is the low half of its dword; past it an
    // odd row's last vector holds zeros already.
#pragma unroll
    for (int d = 0; d < 4; ++d) v[d] = left == 2 * d + 1 ? r.last : v[d];
  }
  return v;
}
template <bool ODD>
__device__ __forceinline__ void half_store(const HalfRow& r, uint32_t off, int left, u32x4 v) {
  if (!ODD) {
    buffer_store_nt(r.dwords, off, v);
  } else if (r.shift == 0) {
    buffer_store_nt(r.dwords, off, v);
    // The last element, alone in its row's last half dword.
    const uint32_t e = left == 1 ? v.x : left == 3 ? v.y : left == 5 ? v.z : v.w;
    const bool here = left > 0 && left < 8;
    __builtin_amdgcn_raw_buffer_store_b16(static_cast<short>(e), r.halves,
                                          here ? off + 2u * (left - 1) : 0xFFFFFFF0u, 0, 0);
  } else {
    // Element 0 in the upper half of the first dword, 1 to 6 in the next
    // three, 7 in the lower half of the fifth.
    typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
    __builtin_amdgcn_raw_buffer_store_b16(static_cast<short>(v.x), r.halves, off + 2u, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b96(
        u32x3{__builtin_amdgcn_alignbit(v.y, v.x, 16), __builtin_amdgcn_alignbit(v.z, v.y, 16),
              __builtin_amdgcn_alignbit(v.w, v.z, 16)},
        r.dwords, off + 4u, 0, kBufferNt);
    __builtin_amdgcn_raw_buffer_store_b16(static_cast<short>(v.w >> 16), r.halves, off + 16u, 0,
                                          0);
  }
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
// Launches READ with the lanes and the loads its rules give a row:
// launch(integral_constant threads, bool_constant vectors).
template <class Launch>
void launch_read(const StreamRule& rule, int64_t rows, int64_t cols, bool vec, Launch&& launch) {
  if (stream_threads(rule, rows, cols) == 1024)  // wide rows
    launch(std::integral_constant<int, 1024>{}, std::true_type{});
  else if (vec || cols >= rule.vectors)
    launch(std::integral_constant<int, 256>{}, std::true_type{});
  else
    launch(std::integral_constant<int, 256>{}, std::false_type{});
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
