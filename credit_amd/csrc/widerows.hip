// Few wide rows in two launches: each row cut into chunks of at most 4096
// columns, one workgroup per chunk.  The first launch leaves every chunk's
// partial sums (fp64) in memory, the second merges its row's and writes the
// outputs.  No workgroup waits for another, so the calls need nothing of the
// device's other work (the SPLIT kernels do), and any width and 4-byte address
// is taken (rows.hpp).  The inputs are read twice, the second time from the L2
// and the MALL while they fit.
// Bound by two launches (6.7-7 us a call from one stream) up to about a million
// elements, by HBM at large ones: the two reads and the write move 6.2 TB/s at
// 256 x 200003.  Against one workgroup per row (registers, then two streamed
// passes) and SPLIT groups, us:
//                       1 x 200003  64 x 40003  384 x 200003  16 x 131072
//   softmax forward       47 -> 7    17 -> 8.6    197 -> 158   10.6 -> 8.0
//   softmax logits bwd   110 -> 7    21 -> 11     373 -> 265   13.9 -> 10.3
//   LayerNorm backward   154 -> 7    38 -> 11     466 -> 260   15.1 -> 10.5
//   quantisation          18 -> 7   9.2 -> 6.6    136 -> 125   11.0 -> 6.8
// and in bf16      1 x 200003  128 x 40003  1000 x 100002  16 x 131072
//   LayerNorm fwd   84 -> 7.8   20 -> 11.7   245 -> 105      9.4 -> 7.7
//   LayerNorm bwd  101 -> 7.3   28 -> 15.5   324 -> 173     12.5 -> 9.2
#include <algorithm>
#include <type_traits>

#include "api_internal.hpp"
#include "common.hpp"
#include "quant_codes.hpp"
#include "rows.hpp"
#include "workspace_cache.hpp"

namespace credit {
namespace {

constexpr int kThreads = 256;
constexpr int kNW = kThreads / kWave;
constexpr int kVpt = 4;
constexpr int kChunk = kThreads * kVpt * 4;  // columns a workgroup holds
constexpr int kMaxParts = kWave;             // one wave merges a row's chunks
constexpr int kValues = 5;                   // fp64 values per chunk
constexpr int kMaxRows = rows::kWideMaxRows;
constexpr float kNegInf = -__builtin_inff();

// Where a workgroup is: its row and its chunk's columns.
struct Place {
  int row, part, parts, c0, n;
  double* out;         // the chunk's partials, [value][part] of the row
  const double* row_partials;
};
__device__ __forceinline__ Place place(double* partials, int cols, int chunk, int parts) {
  Place p;
  p.row = blockIdx.y;
  p.part = blockIdx.x;
  p.parts = parts;
  p.c0 = p.part * chunk;
  p.n = cols - p.c0 < chunk ? cols - p.c0 : chunk;
  double* r = partials + static_cast<size_t>(p.row) * kValues * parts;
  p.out = r + p.part;
  p.row_partials = r;
  return p;
}
template <class T>
__device__ __forceinline__ buffer_rsrc_t chunk_rsrc(const T* base, const Place& p, int cols) {
  return make_rsrc(base + static_cast<size_t>(p.row) * cols + p.c0,
                   static_cast<uint32_t>(p.n * sizeof(T)));
}
__device__ __forceinline__ void chunk_load(f32x4 (&v)[kVpt], buffer_rsrc_t r) {
#pragma unroll
  for (int k = 0; k < kVpt; ++k)
    v[k] = __builtin_bit_cast(f32x4, buffer_load(r, (threadIdx.x + k * kThreads) * 16u));
}
// Elements of the chunk from the lane's k-th vector on.
__device__ __forceinline__ int left_of(const Place& p, int k) {
  return p.n - 4 * static_cast<int>(threadIdx.x + k * kThreads);
}
// Value k of the row's chunks, one per lane (`none` past the last).
__device__ __forceinline__ double partial(const Place& p, int k, double none) {
  const int lane = threadIdx.x & (kWave - 1);
  return lane < p.parts ? p.row_partials[k * p.parts + lane] : none;
}

__device__ __forceinline__ float max4(f32x4 v) {
  return fmax_nan(fmax_nan(v.x, v.y), fmax_nan(v.z, v.w));
}
__device__ __forceinline__ double rescale(double a, double b) {
  return a == -__builtin_inf() ? 0.0 : ::exp(a - b);
}

// ------------------------------------------------------------- softmax ----
// Partials: max m, s = sum e^(x - m), t = sum e^(x - m) dy (logits backward);
// t = sum p dy (backward).
template <WideSoftmax OP>
__global__ __launch_bounds__(kThreads) void softmax_chunks_kernel(
    const float* __restrict__ a, const float* __restrict__ dy, double* __restrict__ partials,
    int cols, int chunk, int parts) {
  __shared__ float mslots[kNW];
  __shared__ double slots[2][kNW];
  const Place p = place(partials, cols, chunk, parts);
  f32x4 v[kVpt], d[kVpt];
  chunk_load(v, chunk_rsrc(a, p, cols));
  if (OP != WideSoftmax::kForward) chunk_load(d, chunk_rsrc(dy, p, cols));
  float m = 0.0f;
  if (OP != WideSoftmax::kBackward) {
    float lm = kNegInf;
#pragma unroll
    for (int k = 0; k < kVpt; ++k)
      lm = fmax_nan(lm, max4(rows::keep4(v[k], left_of(p, k), kNegInf)));
    m = rows::block_max<kNW>(lm, mslots);
  }
  double s = 0.0, t = 0.0;
#pragma unroll
  for (int k = 0; k < kVpt; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float w = v[k][e];
      if (OP != WideSoftmax::kBackward) {
        w = m == kNegInf || left_of(p, k) <= e ? 0.0f : exp_accurate(w - m);
        s += w;
      }
      if (OP != WideSoftmax::kForward) t += static_cast<double>(w * d[k][e]);
    }
  rows::block_sum2<kNW>(s, t, slots);
  if (threadIdx.x == 0) {
    p.out[0] = m;
    p.out[p.parts] = s;
    p.out[2 * p.parts] = t;
  }
}

template <WideSoftmax OP>
__global__ __launch_bounds__(kThreads) void softmax_outputs_kernel(
    const float* __restrict__ a, const float* __restrict__ dy, float* __restrict__ out,
    float* __restrict__ rowmax, float* __restrict__ lse, double* __restrict__ partials, int cols,
    int chunk, int parts) {
  const Place p = place(partials, cols, chunk, parts);
  f32x4 v[kVpt], d[kVpt];
  chunk_load(v, chunk_rsrc(a, p, cols));
  if (OP != WideSoftmax::kForward) chunk_load(d, chunk_rsrc(dy, p, cols));
  float m = 0.0f, inv_s = 1.0f, dot = 0.0f;
  if (OP != WideSoftmax::kBackward) {
    const double mi = partial(p, 0, -__builtin_inf()), si = partial(p, 1, 0.0);
    m = wave_reduce(static_cast<float>(mi), MaxOp{});
    const double f = rescale(mi, m);
    const double s = wave_reduce_sum_f64(si == 0.0 ? 0.0 : si * f);
    inv_s = static_cast<float>(1.0 / s);
    if (OP == WideSoftmax::kLogits)
      dot = static_cast<float>(wave_reduce_sum_f64(partial(p, 2, 0.0) * f) / s);
    if (OP == WideSoftmax::kForward && p.part == 0 && threadIdx.x == 0) {
      rowmax[p.row] = m;
      lse[p.row] = static_cast<float>(static_cast<double>(m) + ::log(s));
    }
  } else {
    dot = static_cast<float>(wave_reduce_sum_f64(partial(p, 2, 0.0)));
  }
  const buffer_rsrc_t r = chunk_rsrc(out, p, cols);
#pragma unroll
  for (int k = 0; k < kVpt; ++k) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float w =
          OP == WideSoftmax::kBackward ? v[k][e] : exp_accurate(v[k][e] - m) * inv_s;
      o[e] = OP == WideSoftmax::kForward ? w : w * (d[k][e] - dot);
    }
    rows::row_store(r, (threadIdx.x + k * kThreads) * 16u, o);
  }
}

// -------------------------------------------------------- quantisation ----
__global__ __launch_bounds__(kThreads) void quant_chunks_kernel(const float* __restrict__ x,
                                                                double* __restrict__ partials,
                                                                int cols, int chunk, int parts) {
  __shared__ float mslots[kNW];
  const Place p = place(partials, cols, chunk, parts);
  f32x4 v[kVpt];
  chunk_load(v, chunk_rsrc(x, p, cols));
  float lm = 0.0f;  // |x| >= 0, and past the chunk x reads 0
#pragma unroll
  for (int k = 0; k < kVpt; ++k)
    lm = fmax_nan(lm, absmax4(v[k]));
  const float m = rows::block_max<kNW>(lm, mslots);
  if (threadIdx.x == 0) p.out[0] = m;
}

__global__ __launch_bounds__(kThreads) void quant_outputs_kernel(
    const float* __restrict__ x, int8_t* __restrict__ q, float* __restrict__ scale,
    double* __restrict__ partials, int cols, int chunk, int parts) {
  const Place p = place(partials, cols, chunk, parts);
  f32x4 v[kVpt];
  chunk_load(v, chunk_rsrc(x, p, cols));
  const float m = wave_reduce(static_cast<float>(partial(p, 0, 0.0)), MaxOp{});
  const float inv = inv_scale(m);
  int8_t* qr = q + static_cast<size_t>(p.row) * cols + p.c0;
#pragma unroll
  for (int k = 0; k < kVpt; ++k) {
    const int left = left_of(p, k);
    int8_t* dst = qr + 4 * (threadIdx.x + k * kThreads);
    if (left >= 4) {
      store_codes(dst, quant4(v[k], inv));
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (left > e) dst[e] = code1(v[k][e], inv);
    }
  }
  if (p.part == 0 && threadIdx.x == 0) scale[p.row] = m / 127.0f;
}

// ----------------------------------------------------------- LayerNorm ----
// 16 elements of a chunk per lane, as floats: four fp32 vectors or two bf16
// ones (ODD: bf16 rows of odd width).
template <class T, bool ODD>
struct Lanes {
  static constexpr int kN = std::is_same_v<T, float> ? 4 : 8;  // elements a vector
  static constexpr int kV = 16 / kN;
  // Elements of the chunk from the lane's k-th vector on.
  __device__ static int left(const Place& p, int k) {
    return p.n - kN * static_cast<int>(threadIdx.x + k * kThreads);
  }
  // Zeros past the chunk.
  __device__ static void load(float (&f)[16], const T* base, size_t at, const Place& p,
                              bool more) {
    if constexpr (kN == 4) {
      const buffer_rsrc_t r = make_rsrc(base + at, static_cast<uint32_t>(p.n) * 4u);
#pragma unroll
      for (int k = 0; k < kV; ++k) {
        const f32x4 v =
            __builtin_bit_cast(f32x4, buffer_load(r, (threadIdx.x + k * kThreads) * 16u));
#pragma unroll
        for (int e = 0; e < 4; ++e) f[4 * k + e] = v[e];
      }
    } else {
      const rows::HalfRow r =
          rows::half_span<ODD, true>(base, at, static_cast<uint32_t>(p.n), more);
#pragma unroll
      for (int k = 0; k < kV; ++k) {
        const u32x4 v =
            rows::half_load<ODD, false>(r, (threadIdx.x + k * kThreads) * 16u, left(p, k));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[8 * k + 2 * e] = bf16_lo(v[e]);
          f[8 * k + 2 * e + 1] = bf16_hi(v[e]);
        }
      }
    }
  }
  __device__ static void store(const float (&f)[16], T* base, size_t at, const Place& p) {
    if constexpr (kN == 4) {
      const buffer_rsrc_t r = make_rsrc(base + at, static_cast<uint32_t>(p.n) * 4u);
#pragma unroll
      for (int k = 0; k < kV; ++k)
        rows::row_store(r, (threadIdx.x + k * kThreads) * 16u,
                        f32x4{f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]});
    } else {
      const rows::HalfRow r =
          rows::half_span<ODD, false>(base, at, static_cast<uint32_t>(p.n), false);
#pragma unroll
      for (int k = 0; k < kV; ++k) {
        u32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = pack_bf16x2(f[8 * k + 2 * e], f[8 * k + 2 * e + 1]);
        rows::half_store<ODD>(r, (threadIdx.x + k * kThreads) * 16u, left(p, k), v);
      }
    }
  }
  __device__ static float first(const T* row) {
    if constexpr (kN == 4)
      return *row;
    else
      return bf16_to_f32(*row);
  }
};

// Partials about the row's first element x0, in fp64: sum(x - x0) and
// sum((x - x0)^2).
template <class L>
__device__ __forceinline__ void deviations(const float (&x)[16], float x0, const Place& p,
                                           double* s1, double* s2) {
  *s1 = *s2 = 0.0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const double c =
        L::left(p, j / L::kN) > j % L::kN ? static_cast<double>(x[j]) - x0 : 0.0;
    *s1 += c;
    *s2 += c * c;
  }
}
struct RowStats {
  double off;  // the mean less x0
  float mean, rstd;
  double rs;
};
// From partials 0 and 1; x0 is kept in the last (dx may be x: not from x).  The
// variance of a row with an infinity or NaN is NaN: 0 in the forward, as in
// layernorm.hip, and NaN in the backward, whose dx is NaN then.
template <bool FORWARD>
__device__ __forceinline__ RowStats row_stats(const Place& p, int cols, float eps) {
  RowStats st;
  st.off = wave_reduce_sum_f64(partial(p, 0, 0.0)) / cols;
  const double var = wave_reduce_sum_f64(partial(p, 1, 0.0)) / cols - st.off * st.off;
  const bool zero = FORWARD ? !(var > 0.0) : var < 0.0;
  st.rs = 1.0 / __builtin_sqrt((zero ? 0.0 : var) + eps);
  st.mean = static_cast<float>(p.row_partials[(kValues - 1) * p.parts] + st.off);
  st.rstd = static_cast<float>(st.rs);
  return st;
}

template <bool ODD>
__global__ __launch_bounds__(kThreads) void layernorm_fwd_chunks_kernel(
    const uint16_t* __restrict__ x, double* __restrict__ partials, int cols, int chunk,
    int parts) {
  using L = Lanes<uint16_t, ODD>;
  __shared__ double slots[2][kNW];
  const Place p = place(partials, cols, chunk, parts);
  const size_t at = static_cast<size_t>(p.row) * cols;
  float v[16];
  L::load(v, x, at + p.c0, p, p.part + 1 < parts);
  float x0 = L::first(x + at);
  if (__builtin_isinf(x0)) x0 = 0.0f;  // the row's mean is infinite, not NaN
  double s1, s2;
  deviations<L>(v, x0, p, &s1, &s2);
  rows::block_sum2<kNW>(s1, s2, slots);
  if (threadIdx.x == 0) {
    p.out[0] = s1;
    p.out[p.parts] = s2;
    p.out[(kValues - 1) * p.parts] = x0;
  }
}

template <bool ODD>
__global__ __launch_bounds__(kThreads) void layernorm_fwd_outputs_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
    const uint16_t* __restrict__ beta, uint16_t* __restrict__ y, float* __restrict__ mean_out,
    float* __restrict__ rstd_out, double* __restrict__ partials, int cols, int chunk, int parts,
    float eps) {
  using L = Lanes<uint16_t, ODD>;
  const Place p = place(partials, cols, chunk, parts);
  const size_t at = static_cast<size_t>(p.row) * cols + p.c0;
  const bool more = p.part + 1 < parts;
  float v[16], g[16], b[16];
  L::load(v, x, at, p, more);
  L::load(g, gamma, p.c0, p, more);
  L::load(b, beta, p.c0, p, more);
  const RowStats st = row_stats<true>(p, cols, eps);
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = (v[j] - st.mean) * st.rstd * g[j] + b[j];
  L::store(v, y, at, p);
  if (p.part == 0 && threadIdx.x == 0) {
    mean_out[p.row] = st.mean;
    rstd_out[p.row] = st.rstd;
  }
}

// Two partials more, with g = dy * gamma: sum g and sum g (x - x0); with d the
// mean less x0, sum g xhat = rstd (sum g (x - x0) - d sum g).
template <class T, bool ODD>
__global__ __launch_bounds__(kThreads) void layernorm_bwd_chunks_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ gamma,
    double* __restrict__ partials, int cols, int chunk, int parts) {
  using L = Lanes<T, ODD>;
  __shared__ double slots[2][2][kNW];
  const Place p = place(partials, cols, chunk, parts);
  const size_t at = static_cast<size_t>(p.row) * cols;
  const bool more = p.part + 1 < parts;
  float v[16], d[16], g[16];
  L::load(v, x, at + p.c0, p, more);
  L::load(d, dy, at + p.c0, p, more);
  L::load(g, gamma, p.c0, p, more);
  const float x0 = L::first(x + at);
  double s1, s2, s3 = 0.0, s4 = 0.0;
  deviations<L>(v, x0, p, &s1, &s2);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const double gg = d[j] * g[j];  // 0 past the chunk
    s3 += gg;
    s4 += gg * (static_cast<double>(v[j]) - x0);
  }
  rows::block_sum2<kNW>(s1, s2, slots[0]);
  rows::block_sum2<kNW>(s3, s4, slots[1]);
  if (threadIdx.x == 0) {
    p.out[0] = s1;
    p.out[p.parts] = s2;
    p.out[2 * p.parts] = s3;
    p.out[3 * p.parts] = s4;
    p.out[(kValues - 1) * p.parts] = x0;
  }
}

template <class T, bool ODD>
__global__ __launch_bounds__(kThreads) void layernorm_bwd_outputs_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ gamma,
    T* __restrict__ dx, double* __restrict__ partials, int cols, int chunk, int parts,
    float eps) {
  using L = Lanes<T, ODD>;
  const Place p = place(partials, cols, chunk, parts);
  const size_t at = static_cast<size_t>(p.row) * cols + p.c0;
  const bool more = p.part + 1 < parts;
  float v[16], d[16], g[16];
  L::load(v, x, at, p, more);
  L::load(d, dy, at, p, more);
  L::load(g, gamma, p.c0, p, more);
  const RowStats st = row_stats<false>(p, cols, eps);
  const double b1 = wave_reduce_sum_f64(partial(p, 2, 0.0));
  const double b2 = wave_reduce_sum_f64(partial(p, 3, 0.0));
  const float mg = static_cast<float>(b1 / cols);
  const float mgx = static_cast<float>(st.rs * (b2 - st.off * b1) / cols);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float xh = (v[j] - st.mean) * st.rstd;
    v[j] = (d[j] * g[j] - mg - xh * mgx) * st.rstd;
  }
  L::store(v, dx, at, p);
}

// ---------------------------------------------------------------- host ----
// The partials live in a buffer per (device, stream) of their own (5 MiB, for
// the first 64 of them): calls that brought no workspace before bring none now
// and share none with the other operations.
using Partials = StreamScratch<ScratchAlloc>;
constexpr size_t kPartialBytes = size_t{kMaxRows} * kMaxParts * kValues * sizeof(double);

struct WidePlan {
  dim3 grid;
  int chunk = 0, parts = 0;
  double* partials = nullptr;
  Partials::Use use;  // held until both launches are made
};

// Where AUTO takes this path (row_rules.hpp).  A caller's workspace is SPLIT's.
bool wide_wanted(const rows::WideRule& rule, const credit_cfg* cfg, int64_t rows, int64_t cols,
                 bool vec) {
  return cfg_variant(cfg) == CREDIT_VARIANT_AUTO && cols <= int64_t{kMaxParts} * kChunk &&
         !(vec && cfg != nullptr && cfg->workspace != nullptr) &&
         rows::wide(rule, rows, cols, vec);
}

// Chunks per row: enough workgroups for three to a CU, at least 1024 columns
// and at most kChunk each.  False: the call's other kernels take it.
bool wide_plan(const rows::WideRule& rule, const credit_cfg* cfg, int64_t rows, int64_t cols,
               bool vec, WidePlan* plan) {
  if (!wide_wanted(rule, cfg, rows, cols, vec)) return false;
  const int64_t least = (cols + kChunk - 1) / kChunk;
  const int64_t most = std::min<int64_t>(kMaxParts, std::max<int64_t>(least, cols / 1024));
  const int64_t want = std::clamp<int64_t>((768 + rows - 1) / rows, least, most);
  plan->chunk = static_cast<int>(((cols + want - 1) / want + 7) / 8 * 8);
  plan->parts = static_cast<int>((cols + plan->chunk - 1) / plan->chunk);
  plan->grid = dim3(static_cast<unsigned>(plan->parts), static_cast<unsigned>(rows));
  static Partials* partials = new Partials(kPartialBytes, 64);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  hipStream_t stream = cfg_stream(cfg);
  if (!keeps_scratch(stream)) return false;
  // Whole vectors run SPLIT under capture, where nothing can be allocated.
  if (vec && prepare_split(cfg) != CREDIT_OK) {
    (void)hipGetLastError();
    return false;
  }
  plan->use = partials->use(dev, stream);
  plan->partials = reinterpret_cast<double*>(plan->use.base);
  return plan->partials != nullptr;
}

template <WideSoftmax OP>
int launch_softmax(const WidePlan& w, const float* a, const float* dy, float* out, float* rowmax,
                   float* lse, int cols, hipStream_t stream) {
  softmax_chunks_kernel<OP><<<w.grid, kThreads, 0, stream>>>(a, dy, w.partials, cols, w.chunk,
                                                             w.parts);
  CREDIT_TRY(check_launch("softmax_chunks_kernel"));
  softmax_outputs_kernel<OP><<<w.grid, kThreads, 0, stream>>>(a, dy, out, rowmax, lse, w.partials,
                                                              cols, w.chunk, w.parts);
  return check_launch("softmax_outputs_kernel");
}

}  // namespace

int wide_softmax(WideSoftmax op, const float* a, const float* dy, float* out, float* rowmax,
                 float* lse, int64_t rows, int64_t cols, bool vec, const credit_cfg* cfg,
                 bool* taken) {
  const rows::WideRule& rule = op == WideSoftmax::kForward    ? rows::kSoftmaxFwdWide
                               : op == WideSoftmax::kBackward ? rows::kSoftmaxBwdWide
                                                              : rows::kLogitsWide;
  WidePlan w;
  if (!(*taken = wide_plan(rule, cfg, rows, cols, vec, &w))) return CREDIT_OK;
  hipStream_t s = cfg_stream(cfg);
  const int c = static_cast<int>(cols);
  switch (op) {
    case WideSoftmax::kForward:
      return launch_softmax<WideSoftmax::kForward>(w, a, dy, out, rowmax, lse, c, s);
    case WideSoftmax::kBackward:
      return launch_softmax<WideSoftmax::kBackward>(w, a, dy, out, rowmax, lse, c, s);
    default:
      return launch_softmax<WideSoftmax::kLogits>(w, a, dy, out, rowmax, lse, c, s);
  }
}

int wide_quant(const float* x, int8_t* q, float* scale, int64_t rows, int64_t cols, bool vec,
               const credit_cfg* cfg, bool* taken) {
  WidePlan w;
  if (!(*taken = wide_plan(rows::kQuantWide, cfg, rows, cols, vec, &w))) return CREDIT_OK;
  hipStream_t s = cfg_stream(cfg);
  const int c = static_cast<int>(cols);
  quant_chunks_kernel<<<w.grid, kThreads, 0, s>>>(x, w.partials, c, w.chunk, w.parts);
  CREDIT_TRY(check_launch("quant_chunks_kernel"));
  quant_outputs_kernel<<<w.grid, kThreads, 0, s>>>(x, q, scale, w.partials, c, w.chunk, w.parts);
  return check_launch("quant_outputs_kernel");
}

template <class T>
int wide_layernorm_bwd(const T* x, const T* dy, const T* gamma, T* dx, int64_t rows, int64_t cols,
                       float eps, bool vec, const credit_cfg* cfg, bool* taken) {
  WidePlan w;
  const rows::WideRule& rule = std::is_same_v<T, float> ? rows::kLnBwdWide : rows::kLnBwdHalfWide;
  if (!(*taken = wide_plan(rule, cfg, rows, cols, vec, &w))) return CREDIT_OK;
  hipStream_t s = cfg_stream(cfg);
  const int c = static_cast<int>(cols);
  const auto launch = [&](auto odd) {
    constexpr bool kOdd = decltype(odd)::value;
    layernorm_bwd_chunks_kernel<T, kOdd><<<w.grid, kThreads, 0, s>>>(x, dy, gamma, w.partials, c,
                                                                     w.chunk, w.parts);
    CREDIT_TRY(check_launch("layernorm_bwd_chunks_kernel"));
    layernorm_bwd_outputs_kernel<T, kOdd><<<w.grid, kThreads, 0, s>>>(
        x, dy, gamma, dx, w.partials, c, w.chunk, w.parts, eps);
    return check_launch("layernorm_bwd_outputs_kernel");
  };
  if constexpr (std::is_same_v<T, uint16_t>) {
    if (cols % 2 != 0) return launch(std::true_type{});
  }
  return launch(std::false_type{});
}
template int wide_layernorm_bwd<float>(const float*, const float*, const float*, float*, int64_t,
                                       int64_t, float, bool, const credit_cfg*, bool*);
template int wide_layernorm_bwd<uint16_t>(const uint16_t*, const uint16_t*, const uint16_t*,
                                          uint16_t*, int64_t, int64_t, float, bool,
                                          const credit_cfg*, bool*);

int wide_layernorm_fwd(const uint16_t* x, const uint16_t* gamma, const uint16_t* beta,
                       uint16_t* y, float* mean, float* rstd, int64_t rows, int64_t cols,
                       float eps, bool vec, const credit_cfg* cfg, bool* taken) {
  WidePlan w;
  if (!(*taken = wide_plan(rows::kLnFwdWide, cfg, rows, cols, vec, &w))) return CREDIT_OK;
  hipStream_t s = cfg_stream(cfg);
  const int c = static_cast<int>(cols);
  const auto launch = [&](auto odd) {
    constexpr bool kOdd = decltype(odd)::value;
    layernorm_fwd_chunks_kernel<kOdd><<<w.grid, kThreads, 0, s>>>(x, w.partials, c, w.chunk,
                                                                  w.parts);
    CREDIT_TRY(check_launch("layernorm_fwd_chunks_kernel"));
    layernorm_fwd_outputs_kernel<kOdd><<<w.grid, kThreads, 0, s>>>(
        x, gamma, beta, y, mean, rstd, w.partials, c, w.chunk, w.parts, eps);
    return check_launch("layernorm_fwd_outputs_kernel");
  };
  return cols % 2 != 0 ? launch(std::true_type{}) : launch(std::false_type{});
}

}  // namespace credit
