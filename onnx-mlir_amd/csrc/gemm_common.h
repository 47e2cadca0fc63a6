// Definitions shared by the int8 GEMM kernels of gemm_kernels.hip and
// gemm_wreg.hip: vector types, the epilogue's parameter block and small device
// helpers.  Device code only; include inside namespace om.
#pragma once

#include "om_kernels.h"

#include <type_traits>
#include <utility>

namespace om {
namespace gemm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
enum : int { kLoadBytes = 0, kLoadAligned = 1, kLoadAny = 2 };
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int BK = kGemmBK;

// Cache policy operand of the buffer stores that carry results: sc1, the
// store is written through to memory when it is issued instead of staying
// dirty in L2 until the kernel ends (2 would be nontemporal, 0 plain).
constexpr int kAuxThrough = 16;
constexpr int kAuxStream = 2;

// Byte offset of 16-byte chunk `c` (0..3) of tile row `r` (row = 64 bytes).
__device__ __forceinline__ int lds_off(int r, int c) {
  return r * BK + ((c ^ ((r >> 2) & 3)) << 4);
}

// A pointer that is the same in every lane, pinned to scalar registers: the
// compiler then addresses memory as (scalar base + 32-bit lane offset) and
// cannot turn base + offset into a per-lane pointer that it advances with
// vector adds.
// A 32-bit lane offset whose widening to 64 bits stays next to its use: hoisted
// out of a loop it would arrive as a 64-bit register pair, and the load would
// then take the per-lane 64-bit address form.
__device__ __forceinline__ uint32_t lane_offset(uint32_t o) {
  asm volatile("" : "+v"(o));
  return o;
}

template <typename T>
__device__ __forceinline__ T *scalar_ptr(T *p) {
  const uint64_t a = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (T *)(((uint64_t)hi << 32) | lo);
}

// Barrier that orders LDS accesses only; global loads already issued keep
// flying across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Where a kernel with the f32 epilogue leaves minimum and maximum of what it
// stored (GemmArgs::y_limits): `out`, null when not asked for; one partial
// pair per block; an arrival counter that is zero between launches.
struct LimitsOut {
  float *out;
  float *part_min, *part_max;
  unsigned *counter;
};

struct EpiParams {
  LimitsOut limits;
  // Kernels that quantize an f32 activation themselves (GemmArgs::X): its
  // minimum and maximum when the caller knows them (GemmArgs::x_limits), so
  // that they are not looked for; null otherwise.
  const float *x_limits;
  const void *a_zp;
  int64_t a_zp_len;
  const void *b_zp;
  int64_t b_zp_len;
  bool need_rowsum;      // B carries an offset: row sums of A' are needed
  const int32_t *colsum;
  const float *a_scale;
  const float *b_scale;
  int64_t b_scale_len;
  const float *y_scale;
  const void *y_zp;
  const float *bias;     // kEpiF32: added after the scaling; null = none
  int64_t bias_len;      // 1 or N
  float floor;           // kEpiF32: relu_floor(whether onnx.Relu follows)
  bool gelu;             // kEpiF32: onnx.Gelu on the result
  void *out;
  bool b_unsigned;
  bool y_unsigned;
  int narrow;
};

// Whether a launch's arguments are few enough for the short way through the launch
// call.  Empty kernels of 64 blocks, one after the other, microseconds a launch:
// structures of 112 bytes 2.8, of 120 bytes 3.5; six pointers 2.9, eight 3.7; a pointer
// and 104 bytes 2.8; two pointers and 72 bytes 2.9, and 88 bytes 3.7; more, up to 320
// bytes, 3.5 - 3.7.  (Grid and block sizes that a kernel reads are 256 bytes of arguments
// behind its own.)
constexpr bool cheap_arguments(size_t bytes, size_t pointers) {
  return (bytes + 15) / 16 * 16 + 8 * pointers < 128;
}
// EpiParams for kernels of a few microseconds (cheap_arguments), without limits of y.
// Fields that no two epilogues need share a place:
//   first   y_scale (kEpiQ8) or bias (kEpiF32)
//   second  y_zp (kEpiQ8) or x_limits (kEpiF32)
// and lengths are told apart as 0, 1 and more (2), which is all that kernels ask.
struct PackedEpi {
  const void *a_zp, *b_zp;
  const int32_t *colsum;
  const float *a_scale, *b_scale;
  const void *first, *second;
  void *out;
  unsigned a_zp_len : 2, b_zp_len : 2, b_scale_len : 2, bias_len : 2;
  unsigned need_rowsum : 1, relu : 1, gelu : 1, b_unsigned : 1, y_unsigned : 1,
      narrow : 1;
};
inline PackedEpi pack_epi(const EpiParams &e, int epi) {
  auto length = [](int64_t n) { return n > 1 ? 2u : (unsigned)n; };
  PackedEpi p = {};
  p.a_zp = e.a_zp;
  p.b_zp = e.b_zp;
  p.colsum = e.colsum;
  p.a_scale = e.a_scale;
  p.b_scale = e.b_scale;
  p.first = epi == kEpiQ8 ? (const void *)e.y_scale : e.bias;
  p.second = epi == kEpiQ8 ? e.y_zp : e.x_limits;
  p.out = e.out;
  p.a_zp_len = length(e.a_zp_len);
  p.b_zp_len = length(e.b_zp_len);
  p.b_scale_len = length(e.b_scale_len);
  p.bias_len = length(e.bias_len);
  p.need_rowsum = e.need_rowsum;
  p.relu = e.floor == 0.0f; // (relu_floor: 0 or a NaN)
  p.gelu = e.gelu;
  p.b_unsigned = e.b_unsigned;
  p.y_unsigned = e.y_unsigned;
  p.narrow = (unsigned)e.narrow;
  return p;
}
static_assert(sizeof(PackedEpi) == 72 && kWrap >= 0 && kWrap < 2 && kSaturate >= 0 &&
              kSaturate < 2);
template <int EPI>
__device__ __forceinline__ EpiParams unpack_epi(const PackedEpi &p) {
  EpiParams e = {};
  e.a_zp = p.a_zp;
  e.b_zp = p.b_zp;
  e.colsum = p.colsum;
  e.a_scale = p.a_scale;
  e.b_scale = p.b_scale;
  if (EPI == kEpiQ8) {
    e.y_scale = (const float *)p.first;
    e.y_zp = p.second;
  } else if (EPI == kEpiF32) {
    e.bias = (const float *)p.first;
    e.x_limits = (const float *)p.second;
  }
  e.out = p.out;
  e.a_zp_len = p.a_zp_len;
  e.b_zp_len = p.b_zp_len;
  e.b_scale_len = p.b_scale_len;
  e.bias_len = p.bias_len;
  e.need_rowsum = p.need_rowsum;
  e.floor = p.relu ? 0.0f : __builtin_nanf("");
  e.gelu = p.gelu;
  e.b_unsigned = p.b_unsigned;
  e.y_unsigned = p.y_unsigned;
  e.narrow = (int)p.narrow;
  return e;
}

template <int EPI>
__device__ __forceinline__ EpiParams unpack_epi(const EpiParams &e) {
  return e;
}
// What the tile kernels are handed; tiles and K steps follow from the sizes.
struct TileArgs {
  const uint8_t *A;
  const int8_t *Bp;
  int M, N, K;
  int steps; // of a part of K (KSplit)
  PackedEpi epi;
};
static_assert(cheap_arguments(sizeof(TileArgs), 0));
__host__ __device__ constexpr int tiles_of(int n, int tile) {
  return (int)(((unsigned)n + tile - 1) / tile);
}
__host__ __device__ constexpr int padded_k(int K) {
  return (int)((K > 0 ? (unsigned)K + BK - 1 : BK) / BK * BK);
}

// Called once by every thread of a block of `nwaves` waves (the waves that are
// still running, in uniform control flow) with the minimum and maximum of the
// elements it stored, NaN ignored (+inf / -inf if it stored none).  The block's
// pair goes to its slot; the block that arrives last folds all slots and
// writes L.out[0..1] (the scheme of DynamicQuantizeLinear's reduction kernel:
// partials as device-scope atomic stores, a ticket drawn after they have been
// acknowledged, the counter put back to zero by the last block).
// lds: 2 * nwaves + 1 words nobody else uses any more; sync: a barrier of the
// calling waves that orders LDS.
template <typename Sync>
__device__ __forceinline__ void block_publish_limits(float lo, float hi,
    const LimitsOut &L, float *lds, int wave, int lane, int nwaves, Sync sync) {
  lo = wave_min(lo);
  hi = wave_max(hi);
  if (lane == 0) {
    lds[wave] = lo;
    lds[nwaves + wave] = hi;
  }
  sync();
  if (wave == 0 && lane == 0) {
    for (int w = 1; w < nwaves; ++w) {
      lo = __builtin_fminf(lo, lds[w]);
      hi = __builtin_fmaxf(hi, lds[nwaves + w]);
    }
    __hip_atomic_store(&L.part_min[blockIdx.x], lo, __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&L.part_max[blockIdx.x], hi, __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): both stores acknowledged
    const unsigned ticket = __hip_atomic_fetch_add(
        L.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    lds[2 * nwaves] = ticket == gridDim.x - 1 ? 1.0f : 0.0f;
  }
  sync();
  if (lds[2 * nwaves] == 0.0f)
    return;
  // the last block to arrive
  lo = __builtin_inff();
  hi = -__builtin_inff();
  for (unsigned i = wave * 64 + lane; i < gridDim.x; i += nwaves * 64) {
    lo = __builtin_fminf(lo, __hip_atomic_load(&L.part_min[i], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT));
    hi = __builtin_fmaxf(hi, __hip_atomic_load(&L.part_max[i], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT));
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  sync(); // (everyone has read the flag)
  if (lane == 0) {
    lds[wave] = lo;
    lds[nwaves + wave] = hi;
  }
  sync();
  if (wave == 0 && lane == 0) {
    for (int w = 1; w < nwaves; ++w) {
      lo = __builtin_fminf(lo, lds[w]);
      hi = __builtin_fmaxf(hi, lds[nwaves + w]);
    }
    L.out[0] = lo;
    L.out[1] = hi;
    __hip_atomic_store(L.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// onnx.Relu as the reference lowers it: max(0, x) with the maximum that
// returns the other operand for a NaN
// (src/Conversion/ONNXToKrnl/Math/Elementwise.cpp:746-754), so NaN -> 0; a
// negative zero becomes +0.
// Done as one maximum per element whether or not a Relu is asked for: against
// `floor` = 0 when it is, and against a NaN when it is not -- that maximum
// (v_max_f32) returns its other operand unchanged, negative zero included, and
// a NaN only when both are.
__device__ __forceinline__ float relu_f32(float f, float floor) {
  return __builtin_fmaxf(f, floor);
}
inline float relu_floor(bool relu) {
  return relu ? 0.0f : __builtin_nanf("");
}

// onnx.Gelu with approximate = "none" as the reference lowers it
// (src/Conversion/ONNXToKrnl/Math/Elementwise.cpp:374-388): (0.5 * x) *
// (1 + erf(x * f32(1 / sqrt 2))), every operation rounded to f32, in this
// order.  The reference's erf is a polynomial approximation that the compiler
// it is built on expands (src/Conversion/KrnlToLLVM/ConvertKrnlToLLVM.cpp:
// 223-225), so no erf reproduces its last bits; this one is
//   erf(m) = sign(m) * (1 - 2^(t * p(t))),  t = min(|m|, 3.925),
// with p of degree 7 fitted (minimax in the error of erf) to log2(erfc(t)) / t
// on [0, 3.925] and the hardware's base-2 exponential: eight multiply-adds, an
// exponential and a subtraction.  Past 3.925, erf rounds to 1 in f32.  Error of
// erf: below 1.5e-7 absolute (0.63 * 2^-22) over the whole line with every
// rounding at its worst, the exponential's one unit in the last place
// included; Gelu needs it absolute, not relative, because the sum 1 + erf is
// what gets multiplied.  Every kernel that applies Gelu calls this function,
// so the result does not depend on which kernel a shape takes.  A NaN gives a
// NaN (through 0.5 * x), +inf gives +inf and -inf gives -inf * 0 = NaN, as the
// formula does.
__device__ __forceinline__ float gelu_erf_f32(float m) {
  const float t = __builtin_fminf(__builtin_fabsf(m), 3.925f);
  float p = -0x1.740ee2p-15f;
  p = __builtin_fmaf(p, t, 0x1.ca2b3ap-12f);
  p = __builtin_fmaf(p, t, -0x1.7ed47ep-10f);
  p = __builtin_fmaf(p, t, -0x1.b09ff2p-11f);
  p = __builtin_fmaf(p, t, 0x1.cfb2b8p-6f);
  p = __builtin_fmaf(p, t, -0x1.302440p-3f);
  p = __builtin_fmaf(p, t, -0x1.d639d0p-1f);
  p = __builtin_fmaf(p, t, -0x1.a0beaap+0f);
  const float e = __builtin_amdgcn_exp2f(p * t);
  return __builtin_copysignf(1.0f - e, m);
}
__device__ __forceinline__ float gelu_f32(float x) {
  const float half_x = 0.5f * x;
  const float e = gelu_erf_f32(x * 0.70710678118654752440f);
  return half_x * (1.0f + e);
}

__device__ __forceinline__ int32_t load_zp_i32(
    const void *p, bool is_unsigned, int64_t i) {
  return is_unsigned ? (int32_t)((const uint8_t *)p)[i]
                     : (int32_t)((const int8_t *)p)[i];
}

// Sum of the 16 int8 values of an MFMA A operand register group (one lane:
// one row, 16 consecutive K bytes).  Kernels add these up over K when the
// epilogue needs rowsum(A'), i.e. when B carries an offset.
// (`ones`: 0x01010101, or 0 to leave the group out.)
__device__ __forceinline__ int32_t frag_rowsum(v4i f, int ones = 0x01010101) {
  int32_t s = __builtin_amdgcn_sdot4(f.x, ones, 0, false);
  s = __builtin_amdgcn_sdot4(f.y, ones, s, false);
  s = __builtin_amdgcn_sdot4(f.z, ones, s, false);
  return __builtin_amdgcn_sdot4(f.w, ones, s, false);
}


// Calls f(std::integral_constant<int, 0>{}) ... f(std::integral_constant<int,
// N - 1>{}): a loop whose index is a compile-time constant in the body.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(
    F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// k_gemm_i8_wreg (gemm_wreg.hip): whether it takes this problem (wreg_ok),
// whether it is the faster kernel for it (wreg_pays), and its launch.
bool wreg_ok(const GemmArgs &g);
bool wreg_pays(int64_t M, int64_t N);
hipError_t launch_gemm_wreg(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode);

// 16 bytes of a row from v, which was read `back` bytes in front of them (so as not
// to run past the end of A): the first `len` (0 .. 16) are the row's, the others
// become those of `fill`.  back < 16, or any number of bytes where len is 0.
__device__ __forceinline__ v4i row_chunk(v4i v, int back, int len, uint64_t fill) {
  uint64_t lo = (uint32_t)v.x | ((uint64_t)(uint32_t)v.y << 32);
  uint64_t hi = (uint32_t)v.z | ((uint64_t)(uint32_t)v.w << 32);
  const int sh = back * 8;
  if (sh >= 64) {
    lo = hi;
    hi = 0;
  }
  const int s1 = sh & 63;
  if (s1) {
    lo = (lo >> s1) | (hi << (64 - s1));
    hi >>= s1;
  }
  const uint64_t mlo =
      len >= 8 ? ~(uint64_t)0 : (((uint64_t)1 << (8 * len)) - 1);
  const uint64_t mhi =
      len >= 16 ? ~(uint64_t)0
                : (len > 8 ? (((uint64_t)1 << (8 * (len - 8))) - 1) : 0);
  lo = (lo & mlo) | (fill & ~mlo);
  hi = (hi & mhi) | (fill & ~mhi);
  return (v4i){(int)(uint32_t)lo, (int)(uint32_t)(lo >> 32), (int)(uint32_t)hi,
      (int)(uint32_t)(hi >> 32)};
}

// Elements between the arrays of the parts of a product split along K.
__host__ __device__ constexpr int64_t part_stride(int64_t M, int64_t N) {
  return (M * N + 3) / 4 * 4;
}
inline int64_t part_stride(const GemmArgs &g) { return part_stride(g.M, g.N); }
inline TileArgs tile_args(const GemmArgs &g, const EpiParams &ep, int epi) {
  return TileArgs{(const uint8_t *)g.A, g.Bp, (int)g.M, (int)g.N, (int)g.K,
      g.split.steps, pack_epi(ep, epi)};
}

// k_gemm_i8_bs and k_gemm_i8_dma_bs (gemm_bs.hip): Bp streamed into registers, K
// a multiple of 16 (128 x 256 tiles: of 256) and A 16-byte aligned; split: one
// of the parts of GemmArgs::split, in 64 x 128 tiles, int32 sums to ep.out.
enum BsTile : int { kBs128x256, kBs64x256, kBs64x128 };
bool bs_ok(const GemmArgs &g, BsTile tile);
hipError_t launch_gemm_bs(hipStream_t st, const GemmArgs &g, const EpiParams &ep,
    int a_mode, BsTile tile);
hipError_t launch_gemm_bs_split(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode);

// k_gemm_i8_skinny (gemm_skinny.hip): up to 64 rows.  skinny_quantizes_rows:
// whether it takes the f32 activation of a fused layer (GemmArgs::X) and
// quantizes it in every block.
bool skinny_ok(int64_t M, int64_t K);
bool skinny_quantizes_rows(int64_t M, int64_t K, const void *x);
hipError_t launch_gemm_skinny(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode);

// k_gemm_i8_flight (gemm_flight.hip): problems that one round of blocks covers,
// K a multiple of 256 up to 1024.  The _dq forms take the f32 activation of a dynamically
// quantized layer (GemmArgs::X) and quantize it in the same launch; the launch
// returns hipErrorNotReady when the exchange between blocks cannot be used
// right now (the caller quantizes with a launch of its own instead).
bool flight_ok(const GemmArgs &g, int a_mode);
hipError_t launch_gemm_flight(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode);
bool flight_quantizes_rows(int64_t M, int64_t K, int64_t N, const void *x);
hipError_t launch_gemm_flight_dq(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, DqlScratch &scratch);

} // namespace gemm
} // namespace om
