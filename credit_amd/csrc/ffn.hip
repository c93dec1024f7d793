// C5: norm-fused FFN on MFMA, bf16 with fp32 accumulation.
//
//   rstd = 1/sqrt(mean_j x^2 + eps)                          (unit RMSNorm weight)
//   h    = bf16(GELU_tanh(rstd * (x @ W1^T)))   shapes of 256-multiples (C5)
//   h    = bf16(GELU_tanh(bf16(x * rstd) @ W1^T))   other shapes (big_shape)
//   out  = bf16(x + h @ W2^T)
//
// On the first the fp32 accumulator of x @ W1^T is multiplied by the row's rstd
// in the epilogue (the row scale commutes with the GEMM), so the normalised
// input is never rounded; on the others the product reads a copy of x scaled
// and rounded to bf16.  Both are the same function up to that
// rounding (the oracle's round_a switch selects either).
//
// No FFN exists in the reference; this is the consumer of the row-norm
// kernels the BASELINE names.  Weights come in the nn.Linear layout
// ([out_features, in_features], K contiguous): W1 [f, d], W2 [d, f], so
// both GEMMs are "A row-major x B K-contiguous" and every MFMA operand
// fragment (8 consecutive k per lane) is one 16-byte LDS read.
// credit_transpose_bf16 converts a [d, f] weight once.
//
// Kernels:
//  1. ffn_rstd_kernel: rstd per row of x (one read of x, 64 MiB at C5).
//  2. GEMM1 with epilogue kEpiGelu: h = bf16(GELU_tanh(acc * rstd[m])); the
//     RMSNorm commutes with the GEMM and is applied as a row scale.
//  3. GEMM2 with epilogue kEpiResidual: out = bf16(acc + x).
// Each GEMM runs on ffn_gemm256_kernel (256 x 256 x 64 tiles, four waves,
// LDS-direct operand loads; the C5 path) or on ffn_gemm_tile_kernel (128 or 256
// x 128 x 64 tiles, K split over workgroups where the tiles leave CUs idle), or
// ffn_gemm_held_kernel (128-tiles, several to a CU), whichever gemm_plan's count
// says is done sooner.  The backward (credit_ffn_rmsnorm_gelu_bwd_bf16) runs
// five GEMMs on the same kernels with its own epilogues.
#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <type_traits>
#include <utility>

#include "api_internal.hpp"
#include "common.hpp"
#include "ffn_plan.hpp"
#include "workspace_cache.hpp"

namespace credit {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

using namespace ffn;

constexpr int kFfnMultiple = 128;  // rows, d and f

// GEMM epilogues.  Forward: kEpiGelu (h = GELU(acc * rstd[m])),
// kEpiResidual (out = acc + x); the training forward's kEpiGeluSave (h =
// GELU(u) to C and u = acc * rstd[m] to C2, both row-major).  Backward
// (credit_ffn_rmsnorm_gelu_bwd_bf16): kEpiUH (u = acc * rstd[m] to C, h =
// GELU(u) transposed to C2), kEpiGeluBwd (du = acc * GELU'(u[m, n]) to C
// and, transposed, to C2), kEpiStore (bf16(acc)), kEpiStoreF32 (acc as fp32
// to Cf).
constexpr int kEpiGelu = 0;
constexpr int kEpiResidual = 1;
constexpr int kEpiUH = 2;
constexpr int kEpiGeluBwd = 3;
constexpr int kEpiStore = 4;
constexpr int kEpiStoreF32 = 5;
constexpr int kEpiGeluSave = 6;
constexpr int kEpiStoreT = 7;  // C^T [N, M] = bf16(acc): the output stored transposed
constexpr int kEpiPartial = 8;  // Cf[slice] = acc as fp32: a K slice's partial sums

// GELU with the tanh approximation, z = sqrt(2/pi) (v + 0.044715 v^3):
// 0.5 (1 + tanh z) = sigmoid(2z), so GELU(v) = v / (1 + e') with
// e' = e^(-2z) = 2^(v t), t = -2 sqrt(2/pi) log2(e) (1 + 0.044715 v^2): one
// hardware exp2 and one hardware reciprocal (about 1 ulp each), no
// cancellation on either side.  On the negative tail e' is large and 1/(1 +
// e') keeps its relative accuracy until e' overflows (v below about -10.5,
// GELU below 4e-38 in magnitude), where rcp(inf) = 0 gives -0; on the
// positive side e' -> 0 and GELU -> v, +inf giving +inf.
constexpr float kGeluC = 0.7978845608028654f;   // sqrt(2/pi)
constexpr float kGeluC2 = 2.302208198144325f;   // 2 sqrt(2/pi) log2(e)
constexpr float kGeluA = 0.044715f;

__device__ __forceinline__ float gelu_tanh(float v) {
  const float t = __builtin_fmaf(-kGeluC2 * kGeluA, v * v, -kGeluC2);
  return v * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * t) + 1.0f);
}

// GELU' needs both s = sigmoid(2z) and r = 1 - s = sigmoid(-2z): with e =
// e^(2z) = 2^(arg), r = 1 / (e + 1) and s = e r, neither cancelling.  The
// exponent is capped at 64 (v above about 6.6), so e stays finite, s rounds
// to 1 and r to 2^-64.
struct GeluParts {
  float r;  // 1 / (e + 1) = 1 - s
  float s;  // sigmoid(2z) = 0.5 (1 + tanh z)
};

__device__ __forceinline__ GeluParts gelu_parts(float v, float v2) {
  const float arg = kGeluC2 * v * __builtin_fmaf(kGeluA, v2, 1.0f);
  const float e = __builtin_amdgcn_exp2f(arg < 64.0f ? arg : 64.0f);
  GeluParts g;
  g.r = __builtin_amdgcn_rcpf(e + 1.0f);
  g.s = e * g.r;
  return g;
}

// d/dv GELU = s + 2 v r s dz/dv, dz/dv = sqrt(2/pi) (1 + 3 * 0.044715 v^2).
__device__ __forceinline__ float gelu_tanh_grad(float v) {
  const float v2 = v * v;
  const GeluParts g = gelu_parts(v, v2);
  return __builtin_fmaf(2.0f * kGeluC * v * g.r * g.s, __builtin_fmaf(3.0f * kGeluA, v2, 1.0f),
                        g.s);
}

// The output values of one element of every epilogue: c goes to C (kEpiStoreF32:
// Cf) and c2 to C2, row-major or transposed as the epilogue says.  s is the
// row scale rstd[m], rv is R[m, n] widened to fp32.
struct EpiValue {
  float c, c2;
};
template <int EPI>
__device__ __forceinline__ EpiValue epilogue_value(float acc, float s, float rv) {
  if constexpr (EPI == kEpiGelu) {
    return {gelu_tanh(acc * s), 0.0f};
  } else if constexpr (EPI == kEpiGeluSave) {
    // The same h as kEpiGelu, and the u the backward's kEpiUH recomputes.
    const float u = acc * s;
    return {gelu_tanh(u), u};
  } else if constexpr (EPI == kEpiResidual) {
    return {acc + rv, 0.0f};
  } else if constexpr (EPI == kEpiUH) {
    const float u = acc * s;
    return {u, gelu_tanh(u)};
  } else if constexpr (EPI == kEpiGeluBwd) {
    const float v = acc * gelu_tanh_grad(rv);
    return {v, v};
  } else {
    return {acc, 0.0f};
  }
}

// Epilogues that read a second [M, N] operand.
template <int EPI>
constexpr bool kEpiReadsR = EPI == kEpiResidual || EPI == kEpiGeluBwd;
// Epilogues that scale row m by scale[m].
template <int EPI>
constexpr bool kEpiScaled = EPI == kEpiGelu || EPI == kEpiGeluSave || EPI == kEpiUH;

__device__ __forceinline__ bf16x8_t scale_bf16x8(bf16x8_t x, float s) {
  const u32x4 v = __builtin_bit_cast(u32x4, x);
  return __builtin_bit_cast(bf16x8_t, u32x4{pack_bf16x2(bf16_lo(v.x) * s, bf16_hi(v.x) * s),
                                            pack_bf16x2(bf16_lo(v.y) * s, bf16_hi(v.y) * s),
                                            pack_bf16x2(bf16_lo(v.z) * s, bf16_hi(v.z) * s),
                                            pack_bf16x2(bf16_lo(v.w) * s, bf16_hi(v.w) * s)});
}

// rstd[m] = 1/sqrt(mean(x[m]^2) + eps); cols % 8 == 0, rows 16-byte aligned.
// With a != nullptr also a = bf16(x * rstd), the row re-read from L2.
__global__ __launch_bounds__(256) void ffn_rstd_kernel(const uint16_t* __restrict__ x,
                                                       float* __restrict__ rstd,
                                                       uint16_t* __restrict__ a, int cols,
                                                       float eps) {
  __shared__ double red[4];
  const u32x4* xr = reinterpret_cast<const u32x4*>(x + static_cast<size_t>(blockIdx.x) * cols);
  const int nvec = cols >> 3;
  float s = 0.0f;
  for (int i = threadIdx.x; i < nvec; i += 256) {
    const u32x4 v = xr[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = bf16_lo(v[e]), hi = bf16_hi(v[e]);
      s += lo * lo + hi * hi;
    }
  }
  const double t = block_reduce_sum_f64<4>(static_cast<double>(s), red);
  const float rs = static_cast<float>(1.0 / __builtin_sqrt(t / cols + eps));
  if (threadIdx.x == 0) rstd[blockIdx.x] = rs;
  if (a == nullptr) return;
  u32x4* ar = reinterpret_cast<u32x4*>(a + static_cast<size_t>(blockIdx.x) * cols);
  for (int i = threadIdx.x; i < nvec; i += 256)
    ar[i] = __builtin_bit_cast(u32x4, scale_bf16x8(__builtin_bit_cast(bf16x8_t, xr[i]), rs));
}

// ----------------------------------------------------- 256 x 256 tiles ---
// The main GEMM: C[m, n] = epi(sum_k A[m, k] * B[n, k]) with 256 x 256 x 64
// tiles per 256-lane workgroup: four waves, one per SIMD.  Wave (wm, wn) of
// the 2 x 2 wave grid owns a 128 x 128 block as 4 x 4
// v_mfma_f32_32x32x16_bf16 tiles (256 fp32 accumulators per lane, held in
// AGPRs).  Measured on the C5 shapes against the eight-wave 256 x 256 x 32
// form with global_load_lds it replaces: +13-17% (1.07 -> 1.23-1.27
// PFLOP/s on GEMM1, bit-identical results); the gain is the K depth of 64
// (every 8 lanes of a load read one whole 128-byte line) and the buffer form
// of the LDS-direct load.
//  - Operand tiles go from global memory straight to LDS with
//    buffer_load_dwordx4 ... lds: a wave instruction writes 1 KiB of LDS
//    (lane l at M0 + 16 l), i.e. 8 rows of 128 bytes.  An operand tile
//    (256 rows x 64 K) is 32 KiB; A has two stages and B three, 160 KiB.
//  - The loads are issued from inline assembly.  The compiler's waitcnt
//    pass cannot tell an LDS-direct load's destination from the fragment
//    reads of the other stage and would wait for every load before every
//    read; here the only waits on the loads are the explicit ones below,
//    which count them (no other vector-memory instruction is in flight in
//    the K loop).
//  - K-step k (64 wide) reads A stage k & 1 and B stage k % 3.  Iteration
//    it runs four sub-steps of 16 MFMAs (k = 16 each), reading the next
//    sub-step's 8 fragments while the current MFMAs issue (interleaving
//    pinned with sched_group_barrier / sched_barrier).  The barrier sits
//    before the last sub-step: own loads of step it+1 landed, then
//    s_barrier publishes step it+1's stages to every wave and proves every
//    wave has read its last fragments of step it.  The last sub-step then
//    reads the first fragments of step it+1.
//  - Loads of step it+2: B (8 per lane) in sub-steps 0-2 of iteration it,
//    3 + 3 + 2 -- its stage (it+2) % 3 was last read in step it-1, before
//    the previous barrier; A (8) in sub-step 3, after the barrier, into A
//    stage it & 1.  Every load thus has at least three sub-steps to land
//    before the wait for it, vmcnt(8) (step it+2's B loads stay in flight).
//    Against two 64 KiB stages, where the last loads of a step had one
//    sub-step: +5.6% on the C5 forward (1291 -> 1363 TFLOP/s, bit-identical
//    outputs).  B's loads spread 2/3/3: the same; 4/4/0 -1%, 0/4/4 -1%,
//    all 8 in sub-step 0: -5%.  Tail steps re-load the last K-step into
//    stages nobody reads again, so the loop body has fixed wait counts.
//  - The barrier is a bare s_barrier after s_waitcnt lgkmcnt(0): a
//    workgroup-scope release fence would also drain the loads in flight.
//  - LDS rows are 128 bytes (64 bf16 of K); 16-byte chunk c of row r sits
//    at position c ^ ((r >> 1) & 7): the 16 lanes of one fragment read
//    (rows r..r+15, one chunk) and of one load's LDS write (rows r, r+1,
//    eight chunks each) hit 16 distinct 4-bank groups.  A load lane picks
//    its global chunk so that it lands at its fixed LDS position.
//   kEpiGelu:     C = bf16(GELU(acc * scale[m]))   (RMSNorm folded in: the
//                 row scale commutes with the GEMM)
//   kEpiResidual: C = bf16(acc + R[m, n])
constexpr int kBigTile = kBig * kBigK * 2;   // one operand tile of a stage, bytes (32 KiB)
constexpr int kBigBRing = 3;                 // B stages (A has two)
constexpr int kBigBBase = 2 * kBigTile;      // B ring after the two A stages
constexpr int kBigLds = (2 + kBigBRing) * kBigTile;  // 160 KiB
// Tile blocks within an XCD: 8 M-tiles x 4 N-tiles run concurrently and
// share their A rows and B columns through that XCD's L2.
constexpr int kGroupM = 8;
constexpr int kBigThreads = 256;

// s_waitcnt vmcnt(n) (gfx9 encoding: vmcnt[3:0] in bits 3:0, vmcnt[5:4] in
// bits 15:14; expcnt and lgkmcnt left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | (0xF << 8) | (0x7 << 4) | (N & 15));
}

// One LDS-direct load: 16 bytes per lane from rsrc at voff + soff into LDS
// at M0 = m0base + QOFF + 16 * lane.  s_nop covers the M0 write -> LDS-DMA
// hazard.  M0 is a reserved register to the compiler, which warns that it
// does not restore a clobbered M0; nothing else in these kernels reads M0
// (no LDS-direct builtins, GWS, s_sendmsg or indexed register moves), so a
// value left by one load is only ever overwritten by the next.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <uint32_t QOFF>
__device__ __forceinline__ void load_to_lds(buffer_rsrc_t rsrc, uint32_t voff, uint32_t m0base,
                                            uint32_t soff) {
  asm volatile(
      "s_add_u32 m0, %2, %3\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, %4 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(m0base), "i"(QOFF), "s"(soff)
      : "memory", "m0", "scc");
}
// The same with the nontemporal hint.
template <uint32_t QOFF>
__device__ __forceinline__ void load_to_lds_nt(buffer_rsrc_t rsrc, uint32_t voff, uint32_t m0base,
                                               uint32_t soff) {
  asm volatile(
      "s_add_u32 m0, %2, %3\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, %4 offen nt lds"
      :
      : "v"(voff), "s"(rsrc), "s"(m0base), "i"(QOFF), "s"(soff)
      : "memory", "m0", "scc");
}
#pragma clang diagnostic pop

// sched_group_barrier masks.
constexpr int kSchedMfma = 0x008;
constexpr int kSchedDsRead = 0x100;

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;

// ds_read_b64_tr_b16 at the LDS location of p (a pointer into smem).
__device__ __forceinline__ bf16x4_t ds_read_tr16(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      reinterpret_cast<lds_bf16x4_t*>((lds_ptr_t)(const_cast<char*>(p))));
}

// Loads per thread per K-step: 16 (8 of A, 8 of B).  Load q of wave w fills
// rows 8 b .. 8 b + 7 of operand q >> 3, b = (q & 7) * 4 + w.
//
// KN: B is stored [K, N] (N contiguous: the [in, out] weight layout, W1
// [d, f] and W2 [f, d]) instead of [N, K].  Its stage is then 64 K-rows of
// 512 bytes (256 columns); load q >= 8 of wave w fills K-rows 8 (q & 7) + 2 w
// and + 1 (one 1 KiB wave instruction), lane l writing 16-byte chunk l % 32
// of row 2 w + l / 32.  Chunk c of K-row r sits at position c ^ 4 (r & 3).
// A B fragment (8 consecutive k of one column per lane) is then gathered by
// two ds_read_b64_tr_b16: within each 16-lane group, result lane 4 a + b
// takes 16-bit word b of the 8-byte pieces addressed by group lanes a,
// a + 4, a + 8, a + 12.  Group lane j addresses K-row k0 + j / 4 and
// columns c0 + 4 (j % 4) .. + 3, so lane j receives column c0 + j at
// K-rows k0 .. k0 + 3 -- the MFMA B operand's layout.  The 32 lanes of one
// half-wave read 4 K-rows x 64 bytes, which the swizzle spreads over all
// 64 banks.

// Clock probe (credit_set_clock_probe): with a non-null `probe`, thread 0 of
// every workgroup adds the shader cycles (s_memtime) and the 100 MHz
// constant-clock ticks (s_memrealtime) between the workgroup's start and its
// end to probe[0] and probe[1] (the start stamps subtracted as it starts, so
// nothing stays live across the kernel); their ratio is the mean shader clock
// the tiles ran at.
__device__ __forceinline__ void clock_probe_add(uint64_t* probe, bool start) {
  if (probe == nullptr || threadIdx.x != 0) return;
  const uint64_t c = __builtin_amdgcn_s_memtime();
  const uint64_t r = __builtin_amdgcn_s_memrealtime();
  __hip_atomic_fetch_add(probe, start ? 0 - c : c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_fetch_add(probe + 1, start ? 0 - r : r, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

template <int EPI, bool KN>
__global__ __launch_bounds__(kBigThreads) void ffn_gemm256_kernel(
    const uint16_t* __restrict__ A, const float* __restrict__ scale,
    const uint16_t* __restrict__ B, const uint16_t* __restrict__ R, uint16_t* __restrict__ C,
    uint16_t* __restrict__ C2, float* __restrict__ Cf, int M, int N, int K,
    uint64_t* __restrict__ probe) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  clock_probe_add(probe, true);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;  // 2 x 2 waves, 128 x 128 each

  // XCD-aware tile order: workgroups are dealt to the 8 XCDs round-robin,
  // so XCD x runs ids x, x + 8, ...; give each XCD a contiguous run of the
  // tile sequence, and walk that run in blocks of kGroupM M-tiles (8 M-tiles
  // x 4 N-tiles run at once per XCD and share A rows and B columns in its L2).
  const int tiles_m = M / kBig, tiles_n = N / kBig;
  const int total = tiles_m * tiles_n;
  const int per_xcd = total / 8;  // host guarantees total % 8 == 0
  const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  const int group = t / (kGroupM * tiles_n);
  const int gm = tiles_m - group * kGroupM < kGroupM ? tiles_m - group * kGroupM : kGroupM;
  const int within = t - group * kGroupM * tiles_n;
  const int tm = group * kGroupM + within % gm;
  const int tn = within / gm;
  const int m0 = tm * kBig, n0 = tn * kBig;
  const int iters = K / kBigK;  // host guarantees an even count >= 2

  // Load addressing.  Lane l of load q reads row 8 b + l / 8 (b as above)
  // and writes LDS chunk l % 8 of it, so it loads logical chunk
  // (l % 8) ^ ((row >> 1) & 7) = (l % 8) ^ ((w & 1) * 4 + l / 16).  The
  // lane-dependent part of the byte offset is one VGPR; row block (q & 7)
  // * 32 rows and the K step go into the scalar offset.
  const buffer_rsrc_t rsrc_a = make_rsrc(A + static_cast<size_t>(m0) * K, 256u * K * 2u);
  // KN: columns n0 .. n0 + 255 of K rows of pitch N (the host keeps K N 2
  // within 32 bits).
  const buffer_rsrc_t rsrc_b =
      KN ? make_rsrc(B + n0, static_cast<uint32_t>((static_cast<size_t>(K - 1) * N + 256) * 2))
         : make_rsrc(B + static_cast<size_t>(n0) * K, 256u * K * 2u);
  const int chunk = (lane & 7) ^ (((wave & 1) << 2) + (lane >> 4));
  const uint32_t voff = static_cast<uint32_t>(((wave * 8 + (lane >> 3)) * K + chunk * 8) * 2);
  const int kn_row = 2 * wave + (lane >> 5);  // K-row of the stage mod 8 (KN loads)
  const uint32_t voff_kn = static_cast<uint32_t>(
      (kn_row * N + (((lane & 31) ^ ((kn_row & 3) << 2)) * 8)) * 2);
  // LDS byte address of smem (an address-space cast; C++ casts do not express it).
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const uint32_t m0_wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
      static_cast<int>(lds0 + wave * 1024)));
  auto load = [&](int k, auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr uint32_t qoff = static_cast<uint32_t>((q & 7) * 4096);
    const int kc = k < iters ? k : iters - 1;  // tail: a harmless re-load
    const int stage_off = q < 8 ? (k & 1) * kBigTile : kBigBBase + (k % kBigBRing) * kBigTile;
    const uint32_t base = static_cast<uint32_t>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(m0_wave + stage_off)));
    const uint32_t soff_nk = static_cast<uint32_t>(kc * kBigK * 2 + (q & 7) * 64 * K);
    const uint32_t soff_kn =
        (static_cast<uint32_t>(kc * kBigK + (q & 7) * 8) * static_cast<uint32_t>(N)) * 2u;
    const uint32_t soff = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
        static_cast<int>(KN && q >= 8 ? soff_kn : soff_nk)));
    if constexpr (q < 8)
      load_to_lds<qoff>(rsrc_a, voff, base, soff);
    else
      load_to_lds<qoff>(rsrc_b, KN ? voff_kn : voff, base, soff);
  };

  // Fragment reads: A rows wm*128 + i*32 + (l & 31), B rows wn*128 + j*32 +
  // (l & 31); K sub-step kk covers logical chunks 2 kk and 2 kk + 1 (lanes
  // 0-31 and 32-63).
  const int fsw = ((lane & 31) >> 1) & 7;
  const int a_frag = (wm * 128 + (lane & 31)) * 128;
  const int b_frag = (wn * 128 + (lane & 31)) * 128;
  // KN fragment j of sub-step kk: group lane j' = l % 16 of group g = (l / 16)
  // % 4 addresses K-row 16 kk + 8 (g / 2) + s (s = j' / 4; + 4 for the
  // second read) and logical chunk 16 wn + 4 j + 2 (g & 1) + (j' / 2) % 2,
  // byte 8 (j' % 2) of it, which sits at position 16 wn + 4 (j ^ s) + ...
  const int kn_g = (lane >> 4) & 3, kn_s = (lane & 15) >> 2;
  const int kn_lane = (8 * (kn_g >> 1) + kn_s) * 512 +
                      (wn * 16 + 2 * (kn_g & 1) + ((lane >> 1) & 1)) * 16 + 8 * (lane & 1);
  struct Frags { bf16x8_t a[4], b[4]; };
  // step: the K-step whose stages are read (A stage step & 1, B stage step % 3).
  auto frag = [&](int step, int kk, int idx) {
    const int c = ((2 * kk + (lane >> 5)) ^ fsw) << 4;
    const char* abase = smem + (step & 1) * kBigTile;
    const char* bbase = smem + kBigBBase + __builtin_amdgcn_readfirstlane(step % kBigBRing) * kBigTile;
    if (KN && idx >= 4) {
      const char* p = bbase + kn_lane + (((idx - 4) ^ kn_s) << 6) + kk * 8192;
      return __builtin_shufflevector(ds_read_tr16(p), ds_read_tr16(p + 2048), 0, 1, 2, 3, 4, 5,
                                     6, 7);
    }
    return idx < 4 ? *reinterpret_cast<const bf16x8_t*>(abase + a_frag + idx * 4096 + c)
                   : *reinterpret_cast<const bf16x8_t*>(bbase + b_frag + (idx - 4) * 4096 + c);
  };
  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // MFMA Mi of a sub-step: fragment read Mi of the next sub-step first (Mi < 8).
  auto mfma = [&]<int Mi>(const Frags& cur, Frags& nxt, int ns, int nkk) {
    if constexpr (Mi < 8) {
      const bf16x8_t v = frag(ns, nkk, Mi);
      if constexpr (Mi < 4)
        nxt.a[Mi] = v;
      else
        nxt.b[Mi - 4] = v;
    }
    acc[Mi >> 2][Mi & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        cur.a[Mi >> 2], cur.b[Mi & 3], acc[Mi >> 2][Mi & 3], 0, 0, 0);
  };
  // A sub-step is four quarters of four MFMAs; load Q0 + j (of step lk)
  // follows quarter j.  Each quarter is a scheduling region of its own (the
  // MFMAs would otherwise drift past the inline-assembly loads and leave
  // them in bursts), with its fragment reads pinned one per MFMA.
  auto sub_step = [&]<int Q0>(const Frags& cur, Frags& nxt, int ns, int nkk, int lk) {
    [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
      (
          [&] {
            constexpr int Qi = Qs;
            [&]<int... Js>(std::integer_sequence<int, Js...>) {
              (mfma.template operator()<4 * Qi + Js>(cur, nxt, ns, nkk), ...);
            }(std::make_integer_sequence<int, 4>{});
            load(lk, std::integral_constant<int, Q0 + Qi>{});
            [&]<int... Js>(std::integer_sequence<int, Js...>) {
              (
                  [&] {
                    constexpr int Mi = 4 * Qi + Js;
                    if constexpr (Mi < 8)  // a KN B fragment is two reads
                      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, KN && Mi >= 4 ? 2 : 1, 0);
                    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                  }(),
                  ...);
            }(std::make_integer_sequence<int, 4>{});
            __builtin_amdgcn_sched_barrier(0);
          }(),
          ...);
    }(std::make_integer_sequence<int, 4>{});
  };

  // Prologue: step 0 whole, then B of step 1 and the first half of its A.
  [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
    (load(0, std::integral_constant<int, Qs>{}), ...);
  }(std::make_integer_sequence<int, 16>{});
  [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
    (load(1, std::integral_constant<int, 8 + Qs>{}), ...);
  }(std::make_integer_sequence<int, 8>{});
  [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
    (load(1, std::integral_constant<int, Qs>{}), ...);
  }(std::make_integer_sequence<int, 4>{});
  wait_vmcnt<12>();  // own loads of step 0 landed
  lds_barrier();
  Frags f0, f1;
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    const bf16x8_t v = frag(0, 0, m);
    if (m < 4)
      f0.a[m] = v;
    else
      f0.b[m - 4] = v;
  }
  // Iteration it computes step it, four loads per sub-step.  Sub-step 0
  // issues the second half of A of step it+1 (its stage (it+1) & 1 was last
  // read in step it-1, before the previous barrier), sub-steps 1-2 B of step
  // it+2 (stage (it+2) % 3, last read in step it-1), and after this
  // iteration's barrier sub-step 3 the first half of A of step it+2 into A
  // stage it & 1, whose reads all precede the barrier.  The wait before the
  // barrier leaves B of step it+2 (8 loads) in flight.
  auto iteration = [&](int it) {
    sub_step.template operator()<4>(f0, f1, it, 1, it + 1);
    sub_step.template operator()<8>(f1, f0, it, 2, it + 2);
    sub_step.template operator()<12>(f0, f1, it, 3, it + 2);
    wait_vmcnt<8>();  // own loads of step it+1 landed
    lds_barrier();
    sub_step.template operator()<0>(f1, f0, it + 1, 0, it + 2);
  };
  for (int it = 0; it < iters; ++it) iteration(it);
  wait_vmcnt<0>();  // the tail re-loads

  // R tile (256 x 256 bf16 = 128 KiB, the whole LDS) for the epilogues that
  // read it: LDS-direct loads, 2 rows of 512 bytes per wave instruction
  // (wave w fills rows 64 w .. 64 w + 63), so the epilogue's per-element
  // reads come from LDS instead of 256 scattered 2-byte global loads per
  // lane.
  const uint16_t* r_tile = reinterpret_cast<const uint16_t*>(smem);
  if constexpr (kEpiReadsR<EPI>) {
    lds_barrier();  // every wave has read its last fragments
    const buffer_rsrc_t rsrc_r = make_rsrc(R + static_cast<size_t>(m0) * N + n0,
                                           static_cast<uint32_t>((255u * N + 256u) * 2u));
    const uint32_t voff_r = static_cast<uint32_t>(((lane >> 5) * N + (lane & 31) * 8) * 2);
    const uint32_t m0_r = static_cast<uint32_t>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(lds0 + wave * 32768)));
    [&]<int... Is>(std::integer_sequence<int, Is...>) {
      (load_to_lds<static_cast<uint32_t>(Is * 1024)>(
           rsrc_r, voff_r, m0_r,
           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane((64 * wave + 2 * Is) * N * 2))),
       ...);
    }(std::make_integer_sequence<int, 32>{});
    wait_vmcnt<0>();
    lds_barrier();
  }
  // R at rows mb .. mb + 3 (mb = the row of accumulator register 4q of tile
  // (i, j)) and the lane's column, by one ds_read_b64_tr_b16: group lane k
  // of each 16-lane group addresses tile row mb + k / 4, columns c0 + 4 (k %
  // 4) .. + 3, so result lane k receives column c0 + k of the four rows --
  // the layout of accumulator registers 4q .. 4q + 3.
  auto r_quad = [&](int i, int j, int q) {
    const int g = lane >> 4, k = lane & 15;
    const int row = wm * 128 + i * 32 + 8 * q + 4 * (g >> 1) + (k >> 2);
    const int col = wn * 128 + j * 32 + 16 * (g & 1) + 4 * (k & 3);
    return ds_read_tr16(reinterpret_cast<const char*>(r_tile) + row * (kBig * 2) + col * 2);
  };

  // Epilogue.  Accumulator register r of lane l holds row
  // 8*(r/4) + 4*(l/32) + r%4 and column l%32 of its 32 x 32 tile.
  if constexpr (EPI == kEpiUH || EPI == kEpiGeluBwd || EPI == kEpiStoreT) {
    // Also (kEpiStoreT: only) stored transposed: registers 4q..4q+3 are four
    // consecutive rows of one column, so each lane writes them as one 8-byte
    // run of C2 (kEpiStoreT: of C).  kEpiGeluBwd with C2 == nullptr skips
    // the transposed copy.
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int mb = m0 + wm * 128 + i * 32 + 8 * q + 4 * (lane >> 5);
          const int n = n0 + wn * 128 + j * 32 + (lane & 31);
          uint32_t t[2];
          bf16x4_t rq;
          if constexpr (EPI == kEpiGeluBwd) rq = r_quad(i, j, q);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int m = mb + e;
            const size_t idx = static_cast<size_t>(m) * N + n;
            float c, ct;
            if (EPI == kEpiUH) {
              c = acc[i][j][4 * q + e] * scale[m];
              ct = gelu_tanh(c);
            } else if (EPI == kEpiGeluBwd) {
              c = ct = acc[i][j][4 * q + e] * gelu_tanh_grad(static_cast<float>(rq[e]));
            } else {
              c = ct = acc[i][j][4 * q + e];
            }
            if (EPI != kEpiStoreT) C[idx] = f32_to_bf16(c);
            const uint32_t b = f32_to_bf16(ct);
            if (e & 1)
              t[e >> 1] |= b << 16;
            else
              t[e >> 1] = b;
          }
          uint16_t* dst = EPI == kEpiStoreT ? C : C2;
          if (EPI != kEpiGeluBwd || C2 != nullptr)
            *reinterpret_cast<uint2*>(dst + static_cast<size_t>(n) * M + mb) = uint2{t[0], t[1]};
        }
    clock_probe_add(probe, false);
    return;
  } else {
  // Registers r and r + 1 (r even) are rows m and m + 1 of one column: both
  // are converted by one packed bf16 conversion and stored as its two halves.
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bf16x4_t rq[4][4];  // [j][q]: R of registers 4q .. 4q + 3 of tile (i, j)
    if constexpr (EPI == kEpiResidual) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) rq[j][q] = r_quad(i, j, q);
    }
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const int m = m0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      constexpr bool kScaled = EPI == kEpiGelu || EPI == kEpiGeluSave;
      const float sc0 = kScaled ? scale[m] : 1.0f;
      const float sc1 = kScaled ? scale[m + 1] : 1.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + wn * 128 + j * 32 + (lane & 31);
        const float a0 = acc[i][j][r], a1 = acc[i][j][r + 1];
        const size_t idx = static_cast<size_t>(m) * N + n;
        if constexpr (EPI == kEpiStoreF32) {
          Cf[idx] = a0;
          Cf[idx + N] = a1;
        } else {
          uint32_t p, p2 = 0;
          if constexpr (EPI == kEpiGelu) {
            p = pack_bf16x2(gelu_tanh(a0 * sc0), gelu_tanh(a1 * sc1));
          } else if constexpr (EPI == kEpiGeluSave) {
            // The same h as kEpiGelu, and the u the backward's kEpiUH recomputes.
            const float u0 = a0 * sc0, u1 = a1 * sc1;
            p = pack_bf16x2(gelu_tanh(u0), gelu_tanh(u1));
            p2 = pack_bf16x2(u0, u1);
          } else if constexpr (EPI == kEpiResidual) {
            p = pack_bf16x2(a0 + static_cast<float>(rq[j][r >> 2][r & 3]),
                            a1 + static_cast<float>(rq[j][r >> 2][(r & 3) + 1]));
          } else {
            static_assert(EPI == kEpiStore, "row-major epilogues only");
            p = pack_bf16x2(a0, a1);
          }
          C[idx] = static_cast<uint16_t>(p);
          C[idx + N] = static_cast<uint16_t>(p >> 16);
          if constexpr (EPI == kEpiGeluSave) {
            C2[idx] = static_cast<uint16_t>(p2);
            C2[idx + N] = static_cast<uint16_t>(p2 >> 16);
          }
        }
      }
    }
  }
  }
  clock_probe_add(probe, false);
}

// The epilogue of registers q .. q + 3 of a 32 x 32 tile: rows mb .. mb + 3 of
// column n.
template <int EPI>
__device__ __forceinline__ void store_quad(const f32x16& acc, int q, const float (&sc)[4],
                                           const uint16_t* R, uint16_t* C, uint16_t* C2, float* Cf,
                                           int mb, int n, int M, int N) {
  const size_t idx = static_cast<size_t>(mb) * N + n;
  EpiValue v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float rv = kEpiReadsR<EPI> ? bf16_to_f32(R[idx + static_cast<size_t>(e) * N]) : 0.0f;
    v[e] = epilogue_value<EPI>(acc[q + e], sc[e], rv);
  }
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    const size_t at = idx + static_cast<size_t>(e) * N;
    if constexpr (EPI == kEpiStoreF32) {
      Cf[at] = v[e].c;
      Cf[at + N] = v[e + 1].c;
    } else if constexpr (EPI != kEpiStoreT) {
      const uint32_t p = pack_bf16x2(v[e].c, v[e + 1].c);
      C[at] = static_cast<uint16_t>(p);
      C[at + N] = static_cast<uint16_t>(p >> 16);
    }
    if constexpr (EPI == kEpiGeluSave) {
      const uint32_t p = pack_bf16x2(v[e].c2, v[e + 1].c2);
      C2[at] = static_cast<uint16_t>(p);
      C2[at + N] = static_cast<uint16_t>(p >> 16);
    }
  }
  const size_t tdx = static_cast<size_t>(n) * M + mb;
  if constexpr (EPI == kEpiStoreT) {
    *reinterpret_cast<uint2*>(C + tdx) =
        uint2{pack_bf16x2(v[0].c, v[1].c), pack_bf16x2(v[2].c, v[3].c)};
  } else if constexpr (EPI == kEpiUH || EPI == kEpiGeluBwd) {
    if (EPI == kEpiUH || C2 != nullptr)
      *reinterpret_cast<uint2*>(C2 + tdx) =
          uint2{pack_bf16x2(v[0].c2, v[1].c2), pack_bf16x2(v[2].c2, v[3].c2)};
  }
}

// ------------------------------------------------- BM x 128 tiles, split K --
// The GEMM of every shape the 256-tile kernel does not fill the chip with:
// BM x 128 x 64 tiles (BM 128 or 256) of four waves in a 2 x 2 grid, wave
// (wm, wn) owning a BM/2 x 64 block as BM/64 x 2 v_mfma_f32_32x32x16_bf16
// tiles, and K cut into `slices` pieces whose fp32 sums are added in slice
// order.
//  - One operand ring for A and B: ST stages of (BM + 128) rows x 64 K, filled
//    by the LDS-direct loads of the 256-tile kernel (the same row swizzle; KN:
//    the stage's B part is 64 K-rows of 256 bytes, chunk c of K-row r at
//    position c ^ 4 (r & 3)).
//  - K-step k reads stage k % ST.  Iteration it runs four sub-steps of k = 16,
//    each reading the next one's fragments while its MFMAs issue.  Before the
//    last sub-step: own loads of step it+1 landed (vmcnt leaves the ST - 2
//    steps behind it in flight), then an LDS-only barrier, after which stage
//    it % ST is free: step it+ST's loads go there, a quarter of them in each
//    of that sub-step and the next iteration's first three (two stages: all in
//    that sub-step).  Steps behind a slice's end are the next slice's first;
//    behind the last slice they re-load its last step into stages nobody reads
//    again.
//  - With few tiles a CU would sit idle or run one long K chain (128 rows x
//    8192 x 28672: 64 tiles on 256 CUs), so gemm_plan cuts K until the units
//    (tiles x slices) fill the chip.  kEpiPartial launches one workgroup per
//    unit, which stores its sums to Cf[slice] for ffn_reduce_kernel; every
//    other EPI covers all slices of its tile in order with the same additions
//    (the loads run on from one slice to the next: 384 x 384 x 7808, 13 slices
//    without scratch, 108 us for the FFN with a prologue each, 95 without),
//    so both forms give the same bits.
//  - B loads carry the nontemporal hint, which leaves the L2 to the A rows
//    that every workgroup of an XCD reads (128 rows x 8192 x 28672: 206 ->
//    196 us; no shape measured slower).
//  - skew: tile column t starts each slice at its (skew t)-th step and wraps
//    around.  A K pitch of a power of two puts the same K-step of every weight
//    row on one channel, and tiles of one wave march in step; apart by one
//    128-byte step each they spread over all channels (230 -> 206 us there).
//    Only where one M-tile covers all rows (weights read once): a product's
//    order of additions must not depend on which side is called M.
//  - RA: the A rows are scaled by scale[m] and rounded to bf16 as their
//    fragments are used.  Twice as slow as reading an A that
//    ffn_rstd_kernel scaled (176 against 87 us for 128 x 28672 x 8192), so it
//    serves calls whose output is in place of x, with no room for that copy.
template <int BM>
constexpr int kTileStageBytes = (BM + kTileN) * kBigK * 2;

template <int EPI, bool KN, int BM, int ST, bool RA>
__global__ __launch_bounds__(256) void ffn_gemm_tile_kernel(
    const uint16_t* __restrict__ A, const float* __restrict__ scale,
    const uint16_t* __restrict__ B, const uint16_t* __restrict__ R, uint16_t* __restrict__ C,
    uint16_t* __restrict__ C2, float* __restrict__ Cf, int M, int N, int K, int slices,
    int skew) {
  constexpr int kStage = kTileStageBytes<BM>;
  constexpr int kBOff = BM * kBigK * 2;    // B after A in a stage
  constexpr int MI = BM / 64;              // 32-row tiles per wave
  constexpr int AL = BM / 32, L = AL + 4;  // loads per wave and step: A, all
  // Loads per sub-step: L3 right behind the barrier, LQ in each of the next
  // three.  With two stages all go behind the barrier: the next wait is three
  // sub-steps away.
  constexpr int L3 = ST == 2 ? L : L / 4, LQ = (L - L3) / 3;
  constexpr int NF = MI + 2;               // fragments per sub-step
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // XCD x runs blocks x, x + 8, ...: a contiguous run of the unit sequence
  // (slice-major), walked in blocks of kGroupM M-tiles as the 256-tile kernel.
  const int tiles_m = M / BM, tiles_n = N / kTileN;
  const int units = static_cast<int>(gridDim.x);
  const int xcd = static_cast<int>(blockIdx.x) % 8, rem = units % 8;
  const int unit = xcd * (units / 8) + (xcd < rem ? xcd : rem) + static_cast<int>(blockIdx.x) / 8;
  const int slice = unit / (tiles_m * tiles_n);
  const int t = unit - slice * tiles_m * tiles_n;
  const int group = t / (kGroupM * tiles_n);
  const int gm = tiles_m - group * kGroupM < kGroupM ? tiles_m - group * kGroupM : kGroupM;
  const int within = t - group * kGroupM * tiles_n;
  const int m0 = (group * kGroupM + within % gm) * BM;
  const int n0 = within / gm * kTileN;
  const int steps = K / kBigK;
  const int s0 = EPI == kEpiPartial ? slice : 0;
  const int s1 = EPI == kEpiPartial ? slice + 1 : slices;
  struct Slice {
    int first, steps, turn;  // K-steps, and the first of them to load
  };
  auto slice_at = [&](int s) {
    Slice r;
    r.first = s * steps / slices;
    r.steps = (s + 1) * steps / slices - r.first;
    r.turn = static_cast<int>(static_cast<uint32_t>(skew * (n0 / kTileN)) %
                              static_cast<uint32_t>(r.steps));
    return r;
  };
  Slice here = slice_at(s0), then = here;  // the slice being summed, and the one behind it
  bool more = false;                       // there is one behind it

  const buffer_rsrc_t rsrc_a =
      make_rsrc(A + static_cast<size_t>(m0) * K, static_cast<uint32_t>(BM) * K * 2u);
  const buffer_rsrc_t rsrc_b =
      KN ? make_rsrc(B + n0,
                     static_cast<uint32_t>((static_cast<size_t>(K - 1) * N + kTileN) * 2))
         : make_rsrc(B + static_cast<size_t>(n0) * K, static_cast<uint32_t>(kTileN) * K * 2u);
  const int chunk = (lane & 7) ^ (((wave & 1) << 2) + (lane >> 4));
  const uint32_t voff = (static_cast<uint32_t>(wave * 8 + (lane >> 3)) * K + chunk * 8) * 2u;
  const uint32_t voff_kn = (static_cast<uint32_t>(wave * 4 + (lane >> 4)) * N +
                            ((lane & 15) ^ ((lane >> 4) << 2)) * 8) * 2u;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const uint32_t m0_wave = static_cast<uint32_t>(
      __builtin_amdgcn_readfirstlane(static_cast<int>(lds0 + wave * 1024)));
  // Load q of the slice's k-th K-step, or past its end the next slice's, into
  // `stage`: A rows 8 (4 q + w) .. + 7 (q < AL), else B rows likewise (KN: K-rows
  // 16 (q - AL) + 4 w .. + 3).
  auto load = [&](int k, int stage, auto qc) {
    constexpr int q = decltype(qc)::value;
    constexpr int qb = q < AL ? q : q - AL;
    constexpr uint32_t qoff = static_cast<uint32_t>(qb * 4096 + (q < AL ? 0 : kBOff));
    const bool behind = EPI != kEpiPartial && more && k >= here.steps;
    const int n = behind ? then.steps : here.steps;
    int kk = behind ? k - here.steps + then.turn
                    : (k < n ? k : n - 1) + here.turn;  // tail: a re-load
    if (kk >= n) kk -= n;
    const uint32_t kc = static_cast<uint32_t>((behind ? then.first : here.first) + kk);
    const uint32_t soff =
        KN && q >= AL ? (kc * kBigK + qb * 16) * static_cast<uint32_t>(N) * 2u
                      : kc * (kBigK * 2) + static_cast<uint32_t>(qb * 64) * static_cast<uint32_t>(K);
    const uint32_t base = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
        static_cast<int>(m0_wave + static_cast<uint32_t>(stage * kStage))));
    const uint32_t so =
        static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(soff)));
    if constexpr (q < AL)
      load_to_lds<qoff>(rsrc_a, voff, base, so);
    else
      load_to_lds_nt<qoff>(rsrc_b, KN ? voff_kn : voff, base, so);
  };

  const int fsw = ((lane & 31) >> 1) & 7;
  const int a_frag = (wm * (BM / 2) + (lane & 31)) * 128;
  const int b_frag = kBOff + (wn * 64 + (lane & 31)) * 128;
  // KN fragment j of sub-step kk: as in the 256-tile kernel, with 256-byte
  // K-rows; the row's swizzle acts on bits 2 and 3 of the chunk, 2 wn + j.
  const int kn_g = (lane >> 4) & 3, kn_s = (lane & 15) >> 2;
  const int kn_lane = kBOff + (8 * (kn_g >> 1) + kn_s) * 256 +
                      (2 * (kn_g & 1) + ((lane >> 1) & 1)) * 16 + 8 * (lane & 1);
  struct Frags { bf16x8_t v[NF]; };  // A fragments, then B
  float a_scale[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
    a_scale[i] = RA ? scale[m0 + wm * (BM / 2) + i * 32 + (lane & 31)] : 1.0f;
  auto frag = [&](int stage, int kk, int idx) {
    const char* base = smem + __builtin_amdgcn_readfirstlane(stage * kStage);
    if (KN && idx >= MI) {
      const char* p = base + kn_lane + (((2 * wn + idx - MI) ^ kn_s) << 6) + kk * 4096;
      return __builtin_shufflevector(ds_read_tr16(p), ds_read_tr16(p + 1024), 0, 1, 2, 3, 4, 5,
                                     6, 7);
    }
    const int c = ((2 * kk + (lane >> 5)) ^ fsw) << 4;
    return *reinterpret_cast<const bf16x8_t*>(
        base + c + (idx < MI ? a_frag + idx * 4096 : b_frag + (idx - MI) * 4096));
  };
  f32x16 acc[MI][2], total[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // One sub-step: 2 MI MFMAs in MI regions of two, region r with fragment
  // reads 2 r and 2 r + 1 of the next sub-step and its share of loads Q0 ..
  // Q0 + NQ - 1 of step lk, each region pinned as in the 256-tile kernel.
  auto sub_step = [&]<int Q0, int NQ>(const Frags& cur, Frags& nxt, int ns, int nkk, int lk, int ls) {
    [&]<int... Rs>(std::integer_sequence<int, Rs...>) {
      (
          [&] {
            constexpr int r = Rs;
            const bf16x8_t a = RA ? scale_bf16x8(cur.v[r], a_scale[r]) : cur.v[r];
            [&]<int... Js>(std::integer_sequence<int, Js...>) {
              (
                  [&] {
                    constexpr int Mi = 2 * r + Js;
                    if constexpr (Mi < NF) nxt.v[Mi] = frag(ns, nkk, Mi);
                    acc[r][Js] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, cur.v[MI + Js],
                                                                         acc[r][Js], 0, 0, 0);
                  }(),
                  ...);
            }(std::make_integer_sequence<int, 2>{});
            [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
              (load(lk, ls, std::integral_constant<int, Q0 + r * NQ / MI + Qs>{}), ...);
            }(std::make_integer_sequence<int, (r + 1) * NQ / MI - r * NQ / MI>{});
            [&]<int... Js>(std::integer_sequence<int, Js...>) {
              (
                  [&] {
                    constexpr int Mi = 2 * r + Js;
                    if constexpr (Mi < NF)
                      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, KN && Mi >= MI ? 2 : 1,
                                                           0);
                    __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                  }(),
                  ...);
            }(std::make_integer_sequence<int, 2>{});
            __builtin_amdgcn_sched_barrier(0);
          }(),
          ...);
    }(std::make_integer_sequence<int, MI>{});
  };
  static_assert(NF <= 2 * MI, "a sub-step's reads fit its regions");

  // Prologue: the first ST - 1 steps whole and the next one's L3 loads; the
  // first step landed before its fragments are read.
#pragma unroll
  for (int k = 0; k < ST - 1; ++k)
    [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
      (load(k, k, std::integral_constant<int, Qs>{}), ...);
    }(std::make_integer_sequence<int, L>{});
  [&]<int... Qs>(std::integer_sequence<int, Qs...>) {
    (load(ST - 1, ST - 1, std::integral_constant<int, Qs>{}), ...);
  }(std::make_integer_sequence<int, L3>{});
  wait_vmcnt<(ST - 2) * L + L3>();
  lds_barrier();
  Frags f0, f1;
#pragma unroll
  for (int m = 0; m < NF; ++m) f0.v[m] = frag(0, 0, m);
  int cur = 0, prev = ST - 1;  // cur = stage of step it, prev of it - 1 and it + ST - 1
  for (int s = s0; s < s1; ++s) {
    more = EPI != kEpiPartial && s + 1 < s1;
    if (more) then = slice_at(s + 1);  // at least 8 steps (gemm_slices), more than the ring holds
    for (int it = 0; it < here.steps; ++it) {
      const int next = cur + 1 == ST ? 0 : cur + 1;
      sub_step.template operator()<L3, LQ>(f0, f1, cur, 1, it + ST - 1, prev);
      sub_step.template operator()<L3 + LQ, LQ>(f1, f0, cur, 2, it + ST - 1, prev);
      sub_step.template operator()<L3 + 2 * LQ, LQ>(f0, f1, cur, 3, it + ST - 1, prev);
      wait_vmcnt<(ST - 2) * L>();  // own loads of step it+1 landed
      lds_barrier();
      sub_step.template operator()<0, L3>(f1, f0, next, 0, it + ST, cur);
      prev = cur;
      cur = next;
    }
    here = then;
    if constexpr (EPI != kEpiPartial) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            total[i][j][r] = s == s0 ? acc[i][j][r] : total[i][j][r] + acc[i][j][r];
            acc[i][j][r] = 0.0f;
          }
    }
  }
  wait_vmcnt<0>();  // the tail re-loads

  // Epilogue.  Registers 4q .. 4q + 3 of tile (i, j) are rows mb .. mb + 3 of
  // column n.
  float* part = Cf + static_cast<size_t>(slice) * M * N;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int mb = m0 + wm * (BM / 2) + i * 32 + 8 * q + 4 * (lane >> 5);
      float sc[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sc[e] = kEpiScaled<EPI> && !RA && scale != nullptr ? scale[mb + e] : 1.0f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn * 64 + j * 32 + (lane & 31);
        if constexpr (EPI == kEpiPartial) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            part[static_cast<size_t>(mb + e) * N + n] = acc[i][j][4 * q + e];
        } else {
          store_quad<EPI>(total[i][j], 4 * q, sc, R, C, C2, Cf, mb, n, M, N);
        }
      }
    }
}

// ------------------------------------------- 128 x 128 tiles, many to a CU --
// More 128-tiles than CUs, unsplit, B [N, K]: one LDS buffer of 36 KiB and the
// next K-step in registers, so that three workgroups share a CU (152 to 165
// registers; kEpiResidual's 175 let two) and cover each other's barriers and
// epilogues, where the ring of ffn_gemm_tile_kernel lets two: 600 tiles of 28 K-steps 55 us against 67 there, 624 of 24 46 against
// 60, 275 of 66 67 against 84, 621 of 18 35 against 48, 1125 of 50 158 against
// 166, 847 of 46 118 against 120 (688 TFLOP/s).  Bound by the LDS reads of 64 x 64 a wave
// and the two barriers of a step.  The same MFMAs in the same order as the
// other kernels' unsplit products: the same bits.
constexpr int kHeldStride = kBigK + 8;  // bf16 per LDS row: 16 bytes of padding spread the banks

template <int EPI>
__global__ __launch_bounds__(256) void ffn_gemm_held_kernel(
    const uint16_t* __restrict__ A, const float* __restrict__ scale,
    const uint16_t* __restrict__ B, const uint16_t* __restrict__ R, uint16_t* __restrict__ C,
    uint16_t* __restrict__ C2, float* __restrict__ Cf, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) uint16_t As[kTileN * kHeldStride];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[kTileN * kHeldStride];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wm = tid >> 7, wn = (tid >> 6) & 1;
  // Consecutive workgroups walk down M: the weight rows stay in the L2.
  const int tiles_m = M / kTileN;
  const int m0 = static_cast<int>(blockIdx.x) % tiles_m * kTileN;
  const int n0 = static_cast<int>(blockIdx.x) / tiles_m * kTileN;

  // Lane t moves 16-byte chunk t % 8 of rows t / 8 + 32 i, of A and of B.
  const int row = tid >> 3, chunk = tid & 7;
  const u32x4* a_src[4];
  const u32x4* b_src[4];
  u32x4 ra[4], rb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const size_t r = row + 32 * i;
    a_src[i] = reinterpret_cast<const u32x4*>(A + (m0 + r) * K) + chunk;
    b_src[i] = reinterpret_cast<const u32x4*>(B + (n0 + r) * K) + chunk;
    ra[i] = *a_src[i];
    rb[i] = *b_src[i];
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t >> 1][t & 1][r] = 0.0f;

  const int steps = K / kBigK;
  for (int k = 0; k < steps; ++k) {
    __syncthreads();  // the last step's fragments are read
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = (row + 32 * i) * kHeldStride + chunk * 8;
      *reinterpret_cast<u32x4*>(As + at) = ra[i];
      *reinterpret_cast<u32x4*>(Bs + at) = rb[i];
    }
    __syncthreads();
    if (k + 1 < steps) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ra[i] = a_src[i][(k + 1) * (kBigK / 8)];
        rb[i] = b_src[i][(k + 1) * (kBigK / 8)];
      }
    }
#pragma unroll
    for (int kk = 0; kk < kBigK; kk += 16) {
      const int at = (lane & 31) * kHeldStride + kk + (lane >> 5) * 8;
      bf16x8_t af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[i] = *reinterpret_cast<const bf16x8_t*>(As + at + (wm * 64 + i * 32) * kHeldStride);
        bf[i] = *reinterpret_cast<const bf16x8_t*>(Bs + at + (wn * 64 + i * 32) * kHeldStride);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
  }

#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int mb = m0 + wm * 64 + i * 32 + 8 * q + 4 * (lane >> 5);
      float sc[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sc[e] = kEpiScaled<EPI> && scale != nullptr ? scale[mb + e] : 1.0f;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        store_quad<EPI>(acc[i][j], 4 * q, sc, R, C, C2, Cf, mb, n0 + wn * 64 + j * 32 + (lane & 31),
                        M, N);
    }
}

// The epilogue of a split GEMM: acc[m, n] = sum over slices, in slice order,
// of part[slice][m][n].  A 64 x 64 block per workgroup, 4 x 4 elements per
// lane (16-byte partial reads, 8-byte stores either way round).
template <int EPI>
__global__ __launch_bounds__(256) void ffn_reduce_kernel(
    const float* __restrict__ part, int slices, const float* __restrict__ scale,
    const uint16_t* __restrict__ R, uint16_t* __restrict__ C, uint16_t* __restrict__ C2,
    float* __restrict__ Cf, int M, int N) {
  const int n = blockIdx.x * 64 + (threadIdx.x & 15) * 4;
  const int m = blockIdx.y * 64 + (threadIdx.x >> 4) * 4;
  const size_t mn = static_cast<size_t>(M) * N;
  f32x4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    acc[e] = *reinterpret_cast<const f32x4*>(part + static_cast<size_t>(m + e) * N + n);
  for (int s = 1; s < slices; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc[e] += *reinterpret_cast<const f32x4*>(part + s * mn + static_cast<size_t>(m + e) * N + n);
  float c2[4][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const size_t idx = static_cast<size_t>(m + e) * N + n;
    const float sc = kEpiScaled<EPI> && scale != nullptr ? scale[m + e] : 1.0f;
    uint2 rw{0, 0};
    if constexpr (kEpiReadsR<EPI>) rw = *reinterpret_cast<const uint2*>(R + idx);
    const float rv[4] = {bf16_lo(rw.x), bf16_hi(rw.x), bf16_lo(rw.y), bf16_hi(rw.y)};
    float c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const EpiValue v = epilogue_value<EPI>(acc[e][k], sc, rv[k]);
      c[k] = v.c;
      c2[e][k] = EPI == kEpiStoreT ? v.c : v.c2;
    }
    if constexpr (EPI == kEpiStoreF32)
      *reinterpret_cast<f32x4*>(Cf + idx) = f32x4{c[0], c[1], c[2], c[3]};
    else if constexpr (EPI != kEpiStoreT)
      *reinterpret_cast<uint2*>(C + idx) =
          uint2{pack_bf16x2(c[0], c[1]), pack_bf16x2(c[2], c[3])};
    if constexpr (EPI == kEpiGeluSave)
      *reinterpret_cast<uint2*>(C2 + idx) =
          uint2{pack_bf16x2(c2[e][0], c2[e][1]), pack_bf16x2(c2[e][2], c2[e][3])};
  }
  if constexpr (EPI == kEpiUH || EPI == kEpiGeluBwd || EPI == kEpiStoreT) {
    uint16_t* dst = EPI == kEpiStoreT ? C : C2;
    if (EPI == kEpiGeluBwd && C2 == nullptr) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      *reinterpret_cast<uint2*>(dst + static_cast<size_t>(n + k) * M + m) =
          uint2{pack_bf16x2(c2[0][k], c2[1][k]), pack_bf16x2(c2[2][k], c2[3][k])};
    }
  }
}

// dst[c, r] = bf16(src[r, c] * scale[r]) (scale == nullptr: a plain copy
// of the bits) for a rows x cols bf16 matrix, through a 64 x 64 LDS tile.
// Full tiles (rows and cols multiples of 64, 16-byte aligned rows) move 16
// bytes per lane on both sides; any other shape takes the element path.
__global__ __launch_bounds__(256) void transpose_bf16_kernel(const uint16_t* __restrict__ src,
                                                             uint16_t* __restrict__ dst,
                                                             int rows, int cols,
                                                             const float* __restrict__ scale,
                                                             int vec) {
  __shared__ uint16_t tile[64][66];  // row stride 132 bytes: column reads spread over banks
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  if (vec) {
    // Load: lane t reads 8 consecutive columns of rows t/8 and t/8 + 32.
    const int lr = threadIdx.x >> 3, lc = (threadIdx.x & 7) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = lr + 32 * h;
      const u32x4 v = *reinterpret_cast<const u32x4*>(src + static_cast<size_t>(r0 + r) * cols + c0 + lc);
      const float sc = scale ? scale[r0 + r] : 1.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t w = v[e];
        if (scale) w = pack_bf16x2(bf16_lo(w) * sc, bf16_hi(w) * sc);
        tile[r][lc + 2 * e] = static_cast<uint16_t>(w & 0xffffu);
        tile[r][lc + 2 * e + 1] = static_cast<uint16_t>(w >> 16);
      }
    }
    __syncthreads();
    // Store: lane t writes 8 consecutive rows of source columns t/8, t/8+32.
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = lr + 32 * h;
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = static_cast<uint32_t>(tile[lc + 2 * e][c]) |
               (static_cast<uint32_t>(tile[lc + 2 * e + 1][c]) << 16);
      *reinterpret_cast<u32x4*>(dst + static_cast<size_t>(c0 + c) * rows + r0 + lc) = o;
    }
    return;
  }
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    const int r = r0 + i, c = c0 + tx;
    if (r < rows && c < cols) {
      uint16_t v = src[static_cast<size_t>(r) * cols + c];
      if (scale) v = f32_to_bf16(bf16_to_f32(v) * scale[r]);
      tile[i][tx] = v;
    }
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int c = c0 + i, r = r0 + tx;
    if (r < rows && c < cols) dst[static_cast<size_t>(c) * rows + r] = tile[tx][i];
  }
}

// dx = dout + rstd * (da - ahat * mean(da * ahat)), ahat = x * rstd: the
// unit-weight RMSNorm backward of the FFN input plus the residual branch.
// One workgroup per row; x, da and dout are read twice (L2-resident rows).
__global__ __launch_bounds__(256) void ffn_dx_kernel(const uint16_t* __restrict__ x,
                                                     const float* __restrict__ rstd,
                                                     const float* __restrict__ da,
                                                     const uint16_t* __restrict__ dout,
                                                     uint16_t* __restrict__ dx, int cols) {
  __shared__ double red[1][4];
  const size_t off = static_cast<size_t>(blockIdx.x) * cols;
  const float rs = rstd[blockIdx.x];
  const int nvec = cols >> 3;
  const u32x4* xv = reinterpret_cast<const u32x4*>(x + off);
  const f32x4* dav = reinterpret_cast<const f32x4*>(da + off);
  float acc = 0.0f;
  for (int i = threadIdx.x; i < nvec; i += 256) {
    const u32x4 v = xv[i];
    const f32x4 d0 = dav[2 * i], d1 = dav[2 * i + 1];
    acc += (bf16_lo(v.x) * d0.x + bf16_hi(v.x) * d0.y) + (bf16_lo(v.y) * d0.z + bf16_hi(v.y) * d0.w) +
           (bf16_lo(v.z) * d1.x + bf16_hi(v.z) * d1.y) + (bf16_lo(v.w) * d1.z + bf16_hi(v.w) * d1.w);
  }
  double dot[1] = {acc};
  block_reduce_sum_f64_multi<4, 1>(dot, red);
  // mean(da * ahat) = rstd * sum(da * x) / cols
  const float c = static_cast<float>(dot[0] * rs / cols);
  const u32x4* gv = reinterpret_cast<const u32x4*>(dout + off);
  u32x4* ov = reinterpret_cast<u32x4*>(dx + off);
  for (int i = threadIdx.x; i < nvec; i += 256) {
    const u32x4 v = xv[i], g = gv[i];
    const f32x4 d0 = dav[2 * i], d1 = dav[2 * i + 1];
    const float dd[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = bf16_lo(g[e]) + rs * (dd[2 * e] - bf16_lo(v[e]) * rs * c);
      const float hi = bf16_hi(g[e]) + rs * (dd[2 * e + 1] - bf16_hi(v[e]) * rs * c);
      o[e] = pack_bf16x2(lo, hi);
    }
    ov[i] = o;
  }
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Sums the 256-tile GEMMs add their clock stamps to (credit_set_clock_probe).
std::atomic<uint64_t*> g_clock_probe{nullptr};

// The GEMM kernels take more dynamic LDS than the default limit; allow it
// once per process and kernel (the attribute belongs to the kernel, not to a
// device).
template <class Kernel>
int allow_lds(Kernel kernel, int bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return e == hipSuccess ? CREDIT_OK
                         : hip_failure(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
}

// Device memory a call's products may use beside its own buffers, for their
// fp32 partial sums.
struct Scratch {
  char* base = nullptr;
  size_t bytes = 0;
};

template <int EPI, bool KN, int BM, int ST, bool RA>
int launch_tile_st(const uint16_t* A, const float* scale, const uint16_t* B, const uint16_t* R,
                uint16_t* C, uint16_t* C2, float* Cf, int M, int N, int K, const GemmPlan& plan,
                hipStream_t stream, const char* name) {
  constexpr int kLds = ST * kTileStageBytes<BM>;
  static const int lds = allow_lds(ffn_gemm_tile_kernel<EPI, KN, BM, ST, RA>, kLds);
  if (lds != CREDIT_OK) return lds;
  const int units = (M / BM) * (N / kTileN) * (EPI == kEpiPartial ? plan.slices : 1);
  ffn_gemm_tile_kernel<EPI, KN, BM, ST, RA><<<dim3(static_cast<unsigned>(units)), dim3(256), kLds,
                                              stream>>>(A, scale, B, R, C, C2, Cf, M, N, K,
                                                        plan.slices, plan.skew);
  return check_launch(name);
}

// Stages by residency: one workgroup per CU takes the LDS whole; more units
// than CUs run two to a CU on two stages each (384 x 3584 x 12416: 128 -> 122
// us for the FFN, 1408 x 2944 x 9856 training step 735 -> 708; a few shapes of
// 1.1 to 1.4 units per CU lose up to 5%).
template <int EPI, bool KN, int BM, bool RA>
int launch_tile(const uint16_t* A, const float* scale, const uint16_t* B, const uint16_t* R,
                uint16_t* C, uint16_t* C2, float* Cf, int M, int N, int K, const GemmPlan& plan,
                hipStream_t stream, const char* name) {
  if constexpr (BM == 256) {
    return launch_tile_st<EPI, KN, BM, 3, RA>(A, scale, B, R, C, C2, Cf, M, N, K, plan, stream,
                                              name);
  } else {
    const int units = (M / BM) * (N / kTileN) * (EPI == kEpiPartial ? plan.slices : 1);
    return units > kGemmCus ? launch_tile_st<EPI, KN, BM, 2, RA>(A, scale, B, R, C, C2, Cf, M, N,
                                                                 K, plan, stream, name)
                            : launch_tile_st<EPI, KN, BM, 4, RA>(A, scale, B, R, C, C2, Cf, M, N,
                                                                 K, plan, stream, name);
  }
}

// C[M, N] = epi(A[M, K] B^T) with B [N, K] (KN false) or [K, N] (KN true);
// M, N and K multiples of 128.  ra: the A rows are scaled by scale and rounded
// as the product runs.  A product that is to be split and whose partial sums
// the scratch does not hold (a smaller caller workspace) runs unsplit, one
// workgroup covering its tile's slices in the same order, with the same bits.
template <int EPI, bool KN = false>
int launch_gemm(const uint16_t* A, const float* scale, const uint16_t* B, const uint16_t* R,
                uint16_t* C, uint16_t* C2, float* Cf, int M, int N, int K, const Scratch& scratch,
                hipStream_t stream, const char* name, bool ra = false) {
  GemmPlan plan = gemm_plan(M, N, K, KN);
  // The weight gradients are formed either way round (M and N swapped).
  if (EPI == kEpiStore || EPI == kEpiStoreT) plan.skew = 0;
  if constexpr (kEpiScaled<EPI>) {
    if (ra)
      return launch_tile<EPI, KN, 128, true>(A, scale, B, R, C, C2, Cf, M, N, K, plan, stream,
                                             name);
  }
  if (plan.big) {
    static const int lds = allow_lds(ffn_gemm256_kernel<EPI, KN>, kBigLds);
    if (lds != CREDIT_OK) return lds;
    ffn_gemm256_kernel<EPI, KN><<<dim3(static_cast<unsigned>((M / kBig) * (N / kBig))),
                                  dim3(kBigThreads), kBigLds, stream>>>(
        A, scale, B, R, C, C2, Cf, M, N, K, g_clock_probe.load(std::memory_order_relaxed));
    return check_launch(name);
  }
  if constexpr (!KN) {
    if (plan.held) {
      const int64_t tiles = int64_t{M / kTileN} * (N / kTileN);
      ffn_gemm_held_kernel<EPI><<<dim3(static_cast<unsigned>(tiles)), dim3(256),
                                  held_extra_lds(tiles, K / kBigK), stream>>>(
          A, scale, B, R, C, C2, Cf, M, N, K);
      return check_launch(name);
    }
  }
  if (plan.slices > 1 &&
      scratch.bytes >= static_cast<size_t>(plan.slices) * M * N * sizeof(float)) {
    float* part = reinterpret_cast<float*>(scratch.base);
    CREDIT_TRY((plan.bm == 256
                    ? launch_tile<kEpiPartial, KN, 256, false>(A, nullptr, B, nullptr, nullptr,
                                                               nullptr, part, M, N, K, plan, stream,
                                                               name)
                    : launch_tile<kEpiPartial, KN, 128, false>(A, nullptr, B, nullptr, nullptr,
                                                               nullptr, part, M, N, K, plan, stream,
                                                               name)));
    ffn_reduce_kernel<EPI><<<dim3(static_cast<unsigned>(N / 64), static_cast<unsigned>(M / 64)),
                             dim3(256), 0, stream>>>(part, plan.slices, scale, R, C, C2, Cf, M, N);
    return check_launch("ffn_reduce_kernel");
  }
  return plan.bm == 256 ? launch_tile<EPI, KN, 256, false>(A, scale, B, R, C, C2, Cf, M, N, K,
                                                           plan, stream, name)
                        : launch_tile<EPI, KN, 128, false>(A, scale, B, R, C, C2, Cf, M, N, K,
                                                           plan, stream, name);
}

// Where a product that rounds a = bf16(x * rstd) first may leave that copy
// until the call writes `out`, [rows, d] bf16 as well; nullptr: out shares
// memory with what the product reads.
uint16_t* copy_room(uint16_t* out, const uint16_t* x, const uint16_t* w1, int64_t rows, int64_t d,
                    int64_t f) {
  const auto apart = [&](const uint16_t* p, int64_t n) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(out), b = reinterpret_cast<uintptr_t>(p);
    return a + static_cast<size_t>(rows * d) * 2 <= b || b + static_cast<size_t>(n) * 2 <= a;
  };
  return apart(x, rows * d) && apart(w1, d * f) ? out : nullptr;
}

// The scaled product u = rstd (x W1^T) with its RMSNorm statistics: rstd, then
// the GEMM over x with rstd in the epilogue, or on the shapes that round
// a = bf16(x * rstd) first over a copy of a at `a` (nullptr: none, the A rows
// are scaled as the product runs).
template <int EPI, bool KN>
int launch_norm_gemm(const uint16_t* x, float* rstd, const uint16_t* w1, uint16_t* C, uint16_t* C2,
                     uint16_t* a, int M, int F, int D, float eps, const Scratch& scratch,
                     hipStream_t stream, const char* name) {
  const bool rounds = !big_shape(M, F, D);
  if (!rounds) a = nullptr;
  ffn_rstd_kernel<<<dim3(M), dim3(256), 0, stream>>>(x, rstd, a, D, eps);
  CREDIT_TRY(check_launch("ffn_rstd_kernel"));
  return launch_gemm<EPI, KN>(a != nullptr ? a : x, a != nullptr ? nullptr : rstd, w1, nullptr, C,
                              C2, nullptr, M, F, D, scratch, stream, name,
                              rounds && a == nullptr);
}

int launch_transpose(const uint16_t* src, uint16_t* dst, int64_t rows, int64_t cols,
                     const float* scale, hipStream_t stream) {
  const int vec = rows % 64 == 0 && cols % 64 == 0 && aligned16(src) && aligned16(dst);
  const dim3 grid(static_cast<unsigned>((cols + 63) / 64), static_cast<unsigned>((rows + 63) / 64));
  transpose_bf16_kernel<<<grid, 256, 0, stream>>>(src, dst, static_cast<int>(rows),
                                                  static_cast<int>(cols), scale, vec);
  return check_launch("transpose_bf16_kernel");
}

// Backward workspace, in order (each region 256-byte aligned): rstd [M]
// fp32; u, du [M, f] and h^T, du^T [f, M] bf16; dout^T, a^T [d, M] bf16;
// da [M, d] fp32.
struct BwdLayout {
  size_t rstd, u, du, ht, dut, doutt, at, da, total;
};
BwdLayout bwd_layout(int64_t M, int64_t d, int64_t f) {
  BwdLayout l;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += align_up(bytes, 256);
    return at;
  };
  l.rstd = take(M * sizeof(float));
  l.u = take(M * f * 2);
  l.du = take(M * f * 2);
  l.ht = take(M * f * 2);
  l.dut = take(M * f * 2);
  l.doutt = take(M * d * 2);
  l.at = take(M * d * 2);
  l.da = take(M * d * sizeof(float));
  l.total = o;
  return l;
}

// Scratch of the whole calls: the most any one of their products uses.
size_t fwd_scratch(int64_t M, int64_t d, int64_t f) {
  return std::max(part_bytes(M, f, d), part_bytes(M, d, f));
}
size_t bwd_scratch(int64_t M, int64_t d, int64_t f) {
  return std::max({part_bytes(M, f, d), part_bytes(d, f, M), part_bytes(M, d, f)});
}

// The training forward brings no workspace and shares none: the partial sums of
// its products, of at most kSlabBytes, live in a buffer per (device, stream) of
// its own, for the first 16 of them; a captured call goes without
// (keeps_scratch), with the same bits.
using TrainScratch = StreamScratch<ScratchAlloc>;
int train_scratch(hipStream_t stream, size_t want, TrainScratch::Use* use, Scratch* out) {
  static TrainScratch* scratch = new TrainScratch(kSlabBytes, 16);
  if (want == 0 || !keeps_scratch(stream)) return CREDIT_OK;
  int dev = 0;
  CREDIT_HIP(hipGetDevice(&dev));
  *use = scratch->use(dev, stream);
  if (use->base != nullptr) *out = Scratch{use->base, want};
  return CREDIT_OK;
}

int check_ffn_shape(int64_t rows, int64_t d, int64_t f) {
  if (rows < 0 || d < 1 || f < 1)
    return set_error(CREDIT_ERR_BAD_SHAPE, "ffn: need rows >= 0, d >= 1, f >= 1");
  if (rows % kFfnMultiple != 0 || d % kFfnMultiple != 0 || f % kFfnMultiple != 0)
    return set_error(CREDIT_ERR_UNSUPPORTED,
                     "ffn: rows, d and f must be multiples of 128 (got %lld, %lld, %lld)",
                     static_cast<long long>(rows), static_cast<long long>(d),
                     static_cast<long long>(f));
  if (rows > (int64_t{1} << 24) || d > (int64_t{1} << 20) || f > (int64_t{1} << 20) ||
      rows * f >= (int64_t{1} << 31) || d * f >= (int64_t{1} << 31) ||
      rows * d >= (int64_t{1} << 31))
    return set_error(CREDIT_ERR_BAD_SHAPE, "ffn: shape too large");
  return CREDIT_OK;
}

}  // namespace

size_t ffn_workspace(int64_t rows, int64_t ffn_dim) {
  return align_up(static_cast<size_t>(rows) * sizeof(float), 256) +
         align_up(static_cast<size_t>(rows) * ffn_dim * sizeof(uint16_t), 256);
}

// What callers are told to bring: the calls' own use plus scratch for their
// products' partial sums, the most there can be since the forward's query does
// not know d (a call runs with any scratch or none).
size_t ffn_workspace_advised(int64_t rows, int64_t ffn_dim) {
  return align_up(ffn_workspace(rows, ffn_dim), 256) + kSlabBytes;
}

size_t ffn_bwd_workspace(int64_t rows, int64_t d, int64_t ffn_dim) {
  return align_up(bwd_layout(rows, d, ffn_dim).total, 256) + bwd_scratch(rows, d, ffn_dim);
}

}  // namespace credit

using namespace credit;

extern "C" int credit_set_clock_probe(uint64_t* sums) {
  if (sums != nullptr) CREDIT_TRY(check_aligned(sums, 8, "sums"));
  g_clock_probe.store(sums, std::memory_order_relaxed);
  return CREDIT_OK;
}

extern "C" int credit_transpose_bf16(const uint16_t* src, uint16_t* dst, int64_t rows,
                                     int64_t cols, const credit_cfg* cfg) {
  CREDIT_TRY(check_row_ptr(src, "src", rows));
  CREDIT_TRY(check_row_ptr(dst, "dst", rows));
  CREDIT_TRY(check_shape(rows, cols, int64_t{1} << 30));
  CREDIT_TRY(check_cfg(cfg));
  if (rows == 0) return CREDIT_OK;
  if (rows > (int64_t{1} << 30))
    return set_error(CREDIT_ERR_BAD_SHAPE, "transpose supports at most 2^30 rows");
  return launch_transpose(src, dst, rows, cols, nullptr, cfg_stream(cfg));
}

namespace credit {
namespace {

// The forward for either weight layout: KN false takes w1 [f, d], w2 [d, f]
// (nn.Linear), KN true w1 [d, f], w2 [f, d] ([in, out]).
template <bool KN>
int ffn_forward(const uint16_t* x, const uint16_t* w1, const uint16_t* w2, uint16_t* out,
                int64_t rows, int64_t d, int64_t f, float eps, const credit_cfg* cfg) {
  CREDIT_TRY(check_row_ptr(x, "x", rows));
  CREDIT_TRY(check_ptr(w1, "w1"));
  CREDIT_TRY(check_ptr(w2, "w2"));
  CREDIT_TRY(check_row_ptr(out, "out", rows));
  CREDIT_TRY(check_cfg(cfg));
  CREDIT_TRY(check_ffn_shape(rows, d, f));
  if (!(eps >= 0.0f)) return set_error(CREDIT_ERR_BAD_CONFIG, "eps must be >= 0");
  if (!aligned16(x) || !aligned16(w1) || !aligned16(w2) || !aligned16(out))
    return set_error(CREDIT_ERR_ALIGNMENT, "ffn: x, w1, w2 and out must be 16-byte aligned");
  if (rows == 0) return CREDIT_OK;
  char* ws = nullptr;
  Scratch scratch;
  uint16_t* a = copy_room(out, x, w1, rows, d, f);
  // In place of x, the copy of a takes scratch too.
  const size_t copy = a != nullptr || big_shape(rows, f, d)
                          ? 0 : align_up(static_cast<size_t>(rows) * d * sizeof(uint16_t), 256);
  const size_t want = copy + fwd_scratch(rows, d, f);
  CREDIT_TRY(acquire_workspace_with(cfg, ffn_workspace(rows, f), want, &ws, &scratch.base,
                                    &scratch.bytes));
  if (copy != 0 && scratch.bytes >= want) {
    a = reinterpret_cast<uint16_t*>(scratch.base);
    scratch = Scratch{scratch.base + copy, scratch.bytes - copy};
  }
  float* rstd = reinterpret_cast<float*>(ws_scratch(ws));
  uint16_t* h = reinterpret_cast<uint16_t*>(
      ws_scratch(ws) + align_up(static_cast<size_t>(rows) * sizeof(float), 256));
  hipStream_t stream = cfg_stream(cfg);
  const int M = static_cast<int>(rows), D = static_cast<int>(d), F = static_cast<int>(f);
  CREDIT_TRY((launch_norm_gemm<kEpiGelu, KN>(x, rstd, w1, h, nullptr, a, M, F, D, eps, scratch,
                                             stream, "ffn gemm1 (gelu)")));
  return launch_gemm<kEpiResidual, KN>(h, nullptr, w2, x, out, nullptr, nullptr, M, D, F, scratch,
                                       stream, "ffn gemm2 (residual)");
}

}  // namespace
}  // namespace credit

extern "C" int credit_ffn_rmsnorm_gelu_bf16(const uint16_t* x, const uint16_t* w1,
                                            const uint16_t* w2, uint16_t* out, int64_t rows,
                                            int64_t d, int64_t f, float eps,
                                            const credit_cfg* cfg) {
  return ffn_forward<false>(x, w1, w2, out, rows, d, f, eps, cfg);
}

namespace credit {
namespace {

template <bool KN>
int ffn_train_forward(const uint16_t* x, const uint16_t* w1, const uint16_t* w2, uint16_t* out,
                      float* rstd, uint16_t* u, uint16_t* h, int64_t rows, int64_t d, int64_t f,
                      float eps, const credit_cfg* cfg) {
  CREDIT_TRY(check_row_ptr(x, "x", rows));
  CREDIT_TRY(check_ptr(w1, "w1"));
  CREDIT_TRY(check_ptr(w2, "w2"));
  CREDIT_TRY(check_row_ptr(out, "out", rows));
  CREDIT_TRY(check_row_ptr(rstd, "rstd", rows));
  CREDIT_TRY(check_row_ptr(u, "u", rows));
  CREDIT_TRY(check_row_ptr(h, "h", rows));
  CREDIT_TRY(check_cfg(cfg));
  CREDIT_TRY(check_ffn_shape(rows, d, f));
  if (!(eps >= 0.0f)) return set_error(CREDIT_ERR_BAD_CONFIG, "eps must be >= 0");
  for (const void* p : {static_cast<const void*>(x), static_cast<const void*>(w1),
                        static_cast<const void*>(w2), static_cast<const void*>(out),
                        static_cast<const void*>(u), static_cast<const void*>(h)})
    if (p && !aligned16(p))
      return set_error(CREDIT_ERR_ALIGNMENT,
                       "ffn training forward: x, w1, w2, out, u and h must be 16-byte aligned");
  if (rows == 0) return CREDIT_OK;
  hipStream_t stream = cfg_stream(cfg);
  TrainScratch::Use use;
  Scratch scratch;
  CREDIT_TRY(train_scratch(stream, fwd_scratch(rows, d, f), &use, &scratch));
  uint16_t* a = copy_room(out, x, w1, rows, d, f);
  const int M = static_cast<int>(rows), D = static_cast<int>(d), F = static_cast<int>(f);
  CREDIT_TRY((launch_norm_gemm<kEpiGeluSave, KN>(x, rstd, w1, h, u, a, M, F, D, eps, scratch,
                                                 stream, "ffn gemm1 (gelu, saving u and h)")));
  return launch_gemm<kEpiResidual, KN>(h, nullptr, w2, x, out, nullptr, nullptr, M, D, F, scratch,
                                       stream, "ffn gemm2 (residual)");
}

}  // namespace
}  // namespace credit

extern "C" int credit_ffn_rmsnorm_gelu_fwd_train_bf16(const uint16_t* x, const uint16_t* w1,
                                                      const uint16_t* w2, uint16_t* out,
                                                      float* rstd, uint16_t* u, uint16_t* h,
                                                      int64_t rows, int64_t d, int64_t f,
                                                      float eps, const credit_cfg* cfg) {
  return ffn_train_forward<false>(x, w1, w2, out, rstd, u, h, rows, d, f, eps, cfg);
}

extern "C" int credit_ffn_rmsnorm_gelu_fwd_train_kn_bf16(const uint16_t* x, const uint16_t* w1,
                                                         const uint16_t* w2, uint16_t* out,
                                                         float* rstd, uint16_t* u, uint16_t* h,
                                                         int64_t rows, int64_t d, int64_t f,
                                                         float eps, const credit_cfg* cfg) {
  return ffn_train_forward<true>(x, w1, w2, out, rstd, u, h, rows, d, f, eps, cfg);
}

extern "C" int credit_ffn_rmsnorm_gelu_kn_bf16(const uint16_t* x, const uint16_t* w1,
                                               const uint16_t* w2, uint16_t* out, int64_t rows,
                                               int64_t d, int64_t f, float eps,
                                               const credit_cfg* cfg) {
  return ffn_forward<true>(x, w1, w2, out, rows, d, f, eps, cfg);
}

namespace credit {
namespace {

// The backward.  With saved == nullptr it recomputes rstd, u and h^T from x
// (one extra GEMM); with the training forward's rstd, u and h it skips that
// GEMM.  Both give the same bits: the saved u and h are the recomputed ones.
// KN false takes the nn.Linear weights (w1 [f, d], w2 [d, f]) and returns
// dW1 [f, d], dW2 [d, f]; KN true the [in, out] weights (w1 [d, f], w2
// [f, d]) and returns dW1 [d, f], dW2 [f, d].  Every GEMM reads the weights,
// dout and the activations in place, as A (K contiguous) or as B in either
// layout; the [in, out] form swaps the operands of the weight-gradient GEMMs
// instead, so it needs neither dout^T nor du^T (only the saved form's dW2,
// whose h^T no GEMM produced, takes dout^T and a transposed store).
struct FfnSaved {
  const float* rstd;
  const uint16_t* u;
  const uint16_t* h;
};

template <bool KN>
int ffn_backward(const uint16_t* x, const uint16_t* w1, const uint16_t* w2,
                 const uint16_t* dout, const FfnSaved* saved, uint16_t* dx, uint16_t* dw1,
                 uint16_t* dw2, int64_t rows, int64_t d, int64_t f, float eps,
                 const credit_cfg* cfg) {
  CREDIT_TRY(check_row_ptr(x, "x", rows));
  CREDIT_TRY(check_ptr(w1, "w1"));
  CREDIT_TRY(check_ptr(w2, "w2"));
  CREDIT_TRY(check_row_ptr(dout, "dout", rows));
  CREDIT_TRY(check_row_ptr(dx, "dx", rows));
  CREDIT_TRY(check_ptr(dw1, "dw1"));
  CREDIT_TRY(check_ptr(dw2, "dw2"));
  CREDIT_TRY(check_cfg(cfg));
  CREDIT_TRY(check_ffn_shape(rows, d, f));
  if (!(eps >= 0.0f)) return set_error(CREDIT_ERR_BAD_CONFIG, "eps must be >= 0");
  if (saved != nullptr) {
    CREDIT_TRY(check_row_ptr(saved->rstd, "rstd", rows));
    CREDIT_TRY(check_row_ptr(saved->u, "u", rows));
    CREDIT_TRY(check_row_ptr(saved->h, "h", rows));
  }
  for (const void* p : {static_cast<const void*>(x), static_cast<const void*>(w1),
                        static_cast<const void*>(w2), static_cast<const void*>(dout),
                        static_cast<const void*>(dx), static_cast<const void*>(dw1),
                        static_cast<const void*>(dw2),
                        static_cast<const void*>(saved ? saved->u : nullptr),
                        static_cast<const void*>(saved ? saved->h : nullptr)})
    if (p && !aligned16(p))
      return set_error(CREDIT_ERR_ALIGNMENT, "ffn backward: every buffer must be 16-byte aligned");
  hipStream_t stream = cfg_stream(cfg);
  if (rows == 0) {
    // No rows: the weight gradients are sums over nothing (zero bits; a
    // fill kernel rather than a memset, so the call can be graph-captured).
    const int64_t words = d * f / 2;  // two bf16 per fp32 word (d, f even)
    const unsigned blocks = static_cast<unsigned>((words + 255) / 256);
    fill_f32_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(reinterpret_cast<float*>(dw1), 0.0f,
                                                             words);
    CREDIT_TRY(check_launch("fill_f32_kernel"));
    fill_f32_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(reinterpret_cast<float*>(dw2), 0.0f,
                                                             words);
    return check_launch("fill_f32_kernel");
  }
  const BwdLayout L = bwd_layout(rows, d, f);
  char* ws = nullptr;
  Scratch scratch;
  CREDIT_TRY(acquire_workspace_with(cfg, L.total, bwd_scratch(rows, d, f), &ws, &scratch.base,
                                    &scratch.bytes));
  char* b = ws_scratch(ws);
  const float* rstd = saved ? saved->rstd : reinterpret_cast<float*>(b + L.rstd);
  const uint16_t* u = saved ? saved->u : reinterpret_cast<uint16_t*>(b + L.u);
  uint16_t* du = reinterpret_cast<uint16_t*>(b + L.du);
  uint16_t* ht = reinterpret_cast<uint16_t*>(b + L.ht);
  uint16_t* dut = reinterpret_cast<uint16_t*>(b + L.dut);
  uint16_t* doutt = reinterpret_cast<uint16_t*>(b + L.doutt);
  uint16_t* at = reinterpret_cast<uint16_t*>(b + L.at);
  float* da = reinterpret_cast<float*>(b + L.da);
  const int M = static_cast<int>(rows), D = static_cast<int>(d), F = static_cast<int>(f);
  // u = (x W1^T) rstd (x W1 for [in, out]), h^T = GELU(u)^T, unless saved; a
  // copy of a passes through da, which the last product writes.
  if (saved == nullptr)
    CREDIT_TRY((launch_norm_gemm<kEpiUH, KN>(x, reinterpret_cast<float*>(b + L.rstd), w1,
                                             reinterpret_cast<uint16_t*>(b + L.u), ht,
                                             reinterpret_cast<uint16_t*>(da), M, F, D, eps,
                                             scratch, stream, "ffn bwd gemm u")));
  // The A operands of the weight gradients in the K-contiguous layout A
  // takes: a^T = bf16(x rstd)^T always, dout^T where no other form reads it.
  if (!KN || saved != nullptr) CREDIT_TRY(launch_transpose(dout, doutt, M, D, nullptr, stream));
  CREDIT_TRY(launch_transpose(x, at, M, D, rstd, stream));
  // du = (dout W2) * GELU'(u) (dout W2^T for [in, out]), with du^T for the
  // nn.Linear dW1 GEMM.
  CREDIT_TRY((launch_gemm<kEpiGeluBwd, !KN>(dout, nullptr, w2, u, du, KN ? nullptr : dut,
                                            nullptr, M, F, D, scratch, stream, "ffn bwd gemm du")));
  if constexpr (!KN) {
    // dW2 [d, f] = dout^T h: h^T [f, M] as the B operand, or the saved h
    // [M, f] read as [K, N].
    if (saved == nullptr)
      CREDIT_TRY(launch_gemm<kEpiStore>(doutt, nullptr, ht, nullptr, dw2, nullptr, nullptr, D, F,
                                        M, scratch, stream, "ffn bwd gemm dw2"));
    else
      CREDIT_TRY((launch_gemm<kEpiStore, true>(doutt, nullptr, saved->h, nullptr, dw2, nullptr,
                                               nullptr, D, F, M, scratch, stream, "ffn bwd gemm dw2")));
    // dW1 [f, d] = du^T a.
    CREDIT_TRY(launch_gemm<kEpiStore>(dut, nullptr, at, nullptr, dw1, nullptr, nullptr, F, D, M,
                                      scratch, stream, "ffn bwd gemm dw1"));
  } else {
    // dW2 [f, d] = h^T dout: h^T as A and dout [M, d] read as [K, N]; from
    // the saved h, (dout^T h)^T with h read as [K, N] and the output stored
    // transposed.
    if (saved == nullptr)
      CREDIT_TRY((launch_gemm<kEpiStore, true>(ht, nullptr, dout, nullptr, dw2, nullptr, nullptr,
                                               F, D, M, scratch, stream, "ffn bwd gemm dw2")));
    else
      CREDIT_TRY((launch_gemm<kEpiStoreT, true>(doutt, nullptr, saved->h, nullptr, dw2, nullptr,
                                                nullptr, D, F, M, scratch, stream, "ffn bwd gemm dw2")));
    // dW1 [d, f] = a^T du: du [M, f] read as [K, N].
    CREDIT_TRY((launch_gemm<kEpiStore, true>(at, nullptr, du, nullptr, dw1, nullptr, nullptr, D, F,
                                             M, scratch, stream, "ffn bwd gemm dw1")));
  }
  // da [M, d] = du W1 (du W1^T for [in, out]), fp32, then dx = dout +
  // RMSNorm backward of da.
  CREDIT_TRY((launch_gemm<kEpiStoreF32, !KN>(du, nullptr, w1, nullptr, nullptr, nullptr, da, M, D,
                                             F, scratch, stream, "ffn bwd gemm da")));
  ffn_dx_kernel<<<dim3(M), dim3(256), 0, stream>>>(x, rstd, da, dout, dx, D);
  return check_launch("ffn_dx_kernel");
}

}  // namespace
}  // namespace credit

extern "C" int credit_ffn_rmsnorm_gelu_bwd_bf16(const uint16_t* x, const uint16_t* w1,
                                                const uint16_t* w2, const uint16_t* dout,
                                                uint16_t* dx, uint16_t* dw1, uint16_t* dw2,
                                                int64_t rows, int64_t d, int64_t f, float eps,
                                                const credit_cfg* cfg) {
  return ffn_backward<false>(x, w1, w2, dout, nullptr, dx, dw1, dw2, rows, d, f, eps, cfg);
}

extern "C" int credit_ffn_rmsnorm_gelu_bwd_saved_bf16(
    const uint16_t* x, const uint16_t* w1, const uint16_t* w2, const uint16_t* dout,
    const float* rstd, const uint16_t* u, const uint16_t* h, uint16_t* dx, uint16_t* dw1,
    uint16_t* dw2, int64_t rows, int64_t d, int64_t f, const credit_cfg* cfg) {
  const FfnSaved saved{rstd, u, h};
  return ffn_backward<false>(x, w1, w2, dout, &saved, dx, dw1, dw2, rows, d, f, 0.0f, cfg);
}

extern "C" int credit_ffn_rmsnorm_gelu_bwd_kn_bf16(const uint16_t* x, const uint16_t* w1,
                                                   const uint16_t* w2, const uint16_t* dout,
                                                   uint16_t* dx, uint16_t* dw1, uint16_t* dw2,
                                                   int64_t rows, int64_t d, int64_t f, float eps,
                                                   const credit_cfg* cfg) {
  return ffn_backward<true>(x, w1, w2, dout, nullptr, dx, dw1, dw2, rows, d, f, eps, cfg);
}

extern "C" int credit_ffn_rmsnorm_gelu_bwd_saved_kn_bf16(
    const uint16_t* x, const uint16_t* w1, const uint16_t* w2, const uint16_t* dout,
    const float* rstd, const uint16_t* u, const uint16_t* h, uint16_t* dx, uint16_t* dw1,
    uint16_t* dw2, int64_t rows, int64_t d, int64_t f, const credit_cfg* cfg) {
  const FfnSaved saved{rstd, u, h};
  return ffn_backward<true>(x, w1, w2, dout, &saved, dx, dw1, dw2, rows, d, f, 0.0f, cfg);
}
