// int8 GEMM for few rows (M <= 64): weight streaming.  What is computed, and
// the layout of Bp, are described at the top of gemm_kernels.hip.
//
// Bound: reading the weights once.  K=4096 N=11008 is 45 MB: 6.4 us at the
// 7.1 TB/s a read-only sweep reaches, plus about 2 us of launch.
//
// Split: a block owns 16 columns (or 32), its 8 waves take contiguous slices of
// K and add their partial sums up in LDS; no barrier in the K loop.  Sixteen
// columns, on v_mfma_i32_16x16x64_i8, because blocks are what the device is
// short of: K=11008 N=4096 gives 256 blocks of 16 columns against 128 of 32, and
// K=4096 N=11008 fills 256 CUs to 2.7 blocks each instead of 1.3.  A wave
// requests a batch of two K steps, waits for it and multiplies; what hides the
// wait is the other waves of the CU (up to 32), and registers are kept for them:
// batches of four steps, or the next batch requested before the wait, leave room
// for fewer and are slower (1 row, K=4096 N=11008: 8.3 us; four steps 9.1, a
// second batch on its way 9.3, both 10.3; 16 waves a block 10.7).  Only up to 4
// rows that arrive quantized, up to 256 blocks, are batches of four ahead
// (launch_rows).
// Streaming (nontemporal) loads of the weights: 10.6 against 10.3 us.
// The epilogue's parameters are requested first and without branches (a wait
// for a zero point in front of the first weights cost 0.5 us).
// Against one 32-column tile per block, four steps a batch and parameters
// loaded behind the K loop (whole fused layer, K=4096 N=11008): 1 row 10.9 -> 8.3
// us, 4 rows 11.5 -> 9.5, 8 rows 13.0 -> 11.5, 16 rows 14.9 -> 13.7, 64 rows
// 19.2 -> 18.1; K=11008 N=4096: 1 row 11.6 -> 9.5, 16 rows 15.8 -> 14.3; 24 rows of
// 1024, N=1024: 6.8 -> 5.6.
//
// DQ: the activation arrives as f32 X[M,K] (at most kSkinnyDqBytes elements) and
// every block quantizes it itself, exactly as DynamicQuantizeLinear would:
// minimum and maximum over all of X, scale and zero point from them, the 8-bit
// values minus 128 into LDS, from where the K loop takes its A operands; the
// first weights are requested before that starts.  Up to 32 Ki elements that
// beats a launch of its own in front (8 rows of 4096: N=4096 6.6 us against 8.1,
// N=11008 10.2 / 11.3; 16 rows of 2048: N=4096 5.8 / 7.3, N=11008 8.6 / 8.2), except
// 17 rows and more of K up to 1024, a multiple of 256, which k_gemm_i8_flight_dq
// could take (32 rows of 1024, N=4096 6.0 / 5.0).
//
// Tried and dropped: one launch in which the first blocks of the grid quantize
// X between them and every block waits for them with its weights already
// requested.  While the weight stream saturates HBM every dependent memory step
// of that chain takes 1.2 to 2 us: 16 rows 15.0 us, 4 rows 12.5, 1 row 11.8.
#include "gemm_common.h"
#include "gemm_epilogue.h"

namespace om {
namespace gemm {

namespace {

constexpr int WAVES = 8;
constexpr int kSkinnyDqBytes = 32768;

// RT row tiles and CT column tiles of T x T, T = 16 or 32 (M <= T * RT).
// DQ: 0, or the float4 of X a thread takes when the block quantizes X itself.
// STG: A rows from global memory pass through a piece of LDS private to the
// wave: a load instruction takes whole rows of the batch (CPR 16-byte chunks
// each, so every cache line it touches is used completely), the MFMA operands
// -- 64 bytes of each of 16 rows -- are read back from there, rows CPR * 16 + 16
// bytes apart to spread them over the banks.  Otherwise the operands are loaded
// directly: the lanes of the rows that are not there fetch nothing.
// ANY: rows of any length, starting at any address (M * K >= 16).  A chunk is read
// where it lies, moved back to end with A where it would run past it; what does
// not belong to the row becomes the byte that stands for 0 behind the shift, in
// the batches that reach the end of K.  (DQ: rows of any length; those in LDS are
// round_up(K, 16) bytes apart.)  Without it such rows were copied by a launch in
// front: layers 13 x 356 x 5568 10.9 -> 3.9 us, 2 x 2380 x 372 10.9 -> 4.1, 15 x
// 8000 x 871 10.2 (K % 16 == 0, as before); int32 12 x 946 x 734 7.6 -> 3.4, 17 x
// 4185 x 1633 7.0 -> 7.0.
struct SkinnyArgs {
  const void *rows; // A, or X (DQ)
  const int8_t *Bp;
  int M, N, K;
  PackedEpi epi;
};
static_assert(cheap_arguments(sizeof(SkinnyArgs), 0));
template <int A_MODE, int EPI, int DQ, int T, int RT, int CT, bool STG, bool ANY>
__global__ __launch_bounds__(WAVES * 64) void k_gemm_i8_skinny(SkinnyArgs args) {
  const uint8_t *__restrict__ A = DQ ? nullptr : (const uint8_t *)args.rows;
  const float *__restrict__ X = DQ ? (const float *)args.rows : nullptr;
  const int8_t *__restrict__ Bp = args.Bp;
  const int M = args.M, N = args.N, K = args.K;
  const EpiParams ep = unpack_epi<EPI>(args.epi);
  static_assert(!DQ || (A_MODE == 2 && !STG), "quantized rows");
  static_assert((T == 16 && CT <= 2) || (T == 32 && CT == 1 && !DQ), "tiles");
  static_assert(!ANY || DQ || STG, "rows of any length");
  constexpr int U = !DQ && !STG ? 4 : 2;    // K steps of a batch
  constexpr int CPR = U * 4;                // 16-byte chunks of a row and batch
  constexpr int RPI = 64 / CPR;             // rows of a load instruction
  constexpr int NLD = STG ? T * RT / RPI : 1;
  constexpr int kPitch = CPR * 16 + 16;
  constexpr int kStageWave = STG ? T * RT * kPitch : 0;
  constexpr int REGS = T * T / 64; // accumulator registers of a tile
  constexpr int SUBS = T / 16;     // MFMAs of a tile and K step
  constexpr int SLOTS = RT * CT * REGS;
  constexpr int kPartBytes = WAVES * SLOTS * 64 * 4;
  // The staged rows, and the rows quantized here, share the memory of the
  // partial sums, which are not written before every wave has left the K loop.
  constexpr int kOwnBytes = DQ ? kSkinnyDqBytes : WAVES * kStageWave;
  constexpr int kLdsBytes = kOwnBytes > kPartBytes ? kOwnBytes : kPartBytes;
  __shared__ __attribute__((aligned(16))) uint8_t lds_raw[kLdsBytes];
  int32_t(*const part)[SLOTS][64] = (int32_t(*)[SLOTS][64])lds_raw;
  __shared__ int32_t rowsum[RT * T]; // of A', over all waves
  __shared__ float s_lo[WAVES], s_hi[WAVES];
  uint8_t *const aq = lds_raw;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & (T - 1); // row of A, column of B
  const int lk = lane / T;       // and 16-byte chunk (of each 64 / SUBS bytes)
  const int KT = (K + BK - 1) / BK;
  const int per = (KT + WAVES - 1) / WAVES;
  const int kt_begin = wave * per < KT ? wave * per : KT;
  const int kt_end = kt_begin + per < KT ? kt_begin + per : KT;

  // The column this thread finishes, and what it is scaled and corrected by:
  // requested first, needed last.
  const int n = blockIdx.x * (T * CT) + (CT == 2 ? ((tid >> 8) & 1) * 16 : 0) + lr;
  const bool col_ok = n < N;
  const int nc = col_ok ? n : 0; // columns past N: computed on column 0, not stored
  constexpr bool A_OFF = (A_MODE != 0);
  const int32_t oa = A_OFF ? 128 : 0;
  const int32_t ob = ep.b_unsigned ? 128 : 0;
  // (No branch around a load: the wait for it would stand there too.  Absent
  // operands are read from colsum, which is always valid, and masked.)
  const bool has_bzp = ep.b_zp_len > 0, has_azp = !DQ && ep.a_zp_len > 0;
  const bool has_bias = EPI == kEpiF32 && ep.bias != nullptr;
  const int32_t bz = load_zp_i32(has_bzp ? ep.b_zp : (const void *)ep.colsum,
      ep.b_unsigned, ep.b_zp_len > 1 ? nc : 0);
  const int32_t az = load_zp_i32(
      has_azp ? ep.a_zp : (const void *)ep.colsum, A_OFF, 0);
  const int32_t cs = ep.colsum[nc];
  const float bias = (has_bias ? ep.bias : (const float *)ep.colsum)
      [has_bias && ep.bias_len > 1 ? nc : 0];
  float bs = 0.0f, as = 0.0f, ys = 1.0f;
  int32_t yz = 0;
  if (EPI != kEpiI32) {
    bs = ep.b_scale[ep.b_scale_len == 1 ? 0 : nc];
    if (!DQ)
      as = ep.a_scale[0];
    if (EPI == kEpiQ8) {
      ys = ep.y_scale[0];
      yz = load_zp_i32(ep.y_zp, ep.y_unsigned, 0);
    }
  }

  if (tid < RT * T)
    rowsum[tid] = 0; // (before the barriers that the additions come after)

  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int NV = DQ > 0 ? DQ : 1;
  f4 v[NV];
  const int nvec = (M * K) >> 2;
  const int P = ANY ? (K + 15) & ~15 : K; // bytes from row to row in LDS (DQ)
  float odd = __builtin_nanf("");          // ANY: of the last M * K % 4 elements
  if (DQ) {
    if (ANY && tid < ((M * K) & 3))
      odd = X[nvec * 4 + tid];
    const f4 *__restrict__ x4 = (const f4 *)X;
    const float nan = __builtin_nanf(""); // neutral for minnum / maxnum
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = j * (WAVES * 64) + tid;
      v[j] = e < nvec ? x4[e] : (f4){nan, nan, nan, nan};
    }
  }

  // Operands of this wave's K steps.  Steps past its slice are sent outside the
  // descriptors and read as zeros (no memory traffic): B' = 0 there.
  constexpr int kOutside = 0x7FFFFFFF;
  const int tile = T * CT == 32 ? (int)blockIdx.x : (int)blockIdx.x >> 1;
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(Bp + (int64_t)tile * KT * 2048), 0, KT * 2048, 0x00020000);
  const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)A, 0, DQ ? 0 : M * K, 0x00020000);
  int bvoff[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
    bvoff[c] = T == 32 ? lane * 16
                       : (lk >> 1) * 1024 +
                             ((lk & 1) * 32 +
                                 (CT == 2 ? c : ((int)blockIdx.x & 1)) * 16 + lr) * 16;

  struct Batch {
    v4i b[U][CT][SUBS];
    v4i a[STG ? NLD : (DQ ? 1 : U)];
  };
  auto request = [&](int kt, Batch &t) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = kt + u;
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int b = 0; b < SUBS; ++b)
          t.b[u][c][b] = __builtin_amdgcn_raw_buffer_load_b128(brsrc,
              s < kt_end ? bvoff[c] + b * 1024 : kOutside,
              s < kt_end ? s * 2048 : 0, 0);
    }
    if (STG) {
      const int s = kt + (lane % CPR) / 4;
      const int k0 = s * BK + (lane & 3) * 16;
      const bool k_in = s < kt_end && k0 < K; // (K % 16 == 0: in or out)
#pragma unroll
      for (int j = 0; j < NLD; ++j) {
        const int row = j * RPI + lane / CPR;
        if (ANY) {
          const uint8_t *const last = A + (M * K - 16);
          const uint8_t *const at = A + (row * K + k0);
          t.a[j] = *(const v4i_any *)(k_in && row < M && at < last ? at : last);
          continue;
        }
        t.a[j] = __builtin_amdgcn_raw_buffer_load_b128(
            arsrc, k_in && row < M ? row * K + k0 : kOutside, 0, 0);
      }
    } else if (!DQ) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k0 = (kt + u) * BK + lk * 16;
        const bool in = lr < M && kt + u < kt_end && k0 < K;
        t.a[u] = __builtin_amdgcn_raw_buffer_load_b128(
            arsrc, in ? lr * K + k0 : kOutside, 0, 0);
      }
    }
  };
  Batch first; // DQ: on its way while the block quantizes its rows
  if (DQ) {
    request(kt_begin, first);
    __builtin_amdgcn_sched_barrier(0);
  }

  float dq_scale = 0.0f;
  int32_t dq_zp = 0;
  if (DQ) {
    float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      lo = __builtin_fminf(__builtin_fminf(lo, v[j].x),
          __builtin_fminf(__builtin_fminf(v[j].y, v[j].z), v[j].w));
      hi = __builtin_fmaxf(__builtin_fmaxf(hi, v[j].x),
          __builtin_fmaxf(__builtin_fmaxf(v[j].y, v[j].z), v[j].w));
    }
    lo = __builtin_fminf(lo, odd);
    hi = __builtin_fmaxf(hi, odd);
    if (ep.x_limits) { // (the same for every thread) known from the layer before
      lo = ep.x_limits[0];
      hi = ep.x_limits[1];
    } else {
      lo = wave_min(lo);
      hi = wave_max(hi);
      if (lane == 0) {
        s_lo[wave] = lo;
        s_hi[wave] = hi;
      }
      lds_barrier();
      lo = s_lo[0];
      hi = s_hi[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) {
        lo = __builtin_fminf(lo, s_lo[w]);
        hi = __builtin_fmaxf(hi, s_hi[w]);
      }
    }
    float zpf;
    dynamic_params(lo, hi, dq_scale, zpf);
    dq_zp = (int32_t)(uint32_t)zpf;
    const float recip = 1.0f / dq_scale;
    auto quantize = [&](auto fast_c) {
      constexpr bool FAST = decltype(fast_c)::value;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int e = j * (WAVES * 64) + tid;
        if (e < nvec) {
          const uint32_t q = quant_pack4<false, true, FAST>(v[j].x, v[j].y,
              v[j].z, v[j].w, dq_scale, dq_scale, dq_scale, dq_scale, recip,
              recip, recip, recip, zpf, zpf, zpf, zpf);
          if (!ANY) {
            ((uint32_t *)aq)[e] = q ^ 0x80808080u;
            continue;
          }
          uint32_t r = (uint32_t)(e * 4) / (uint32_t)K;
          uint32_t c = (uint32_t)(e * 4) - r * (uint32_t)K;
          if ((K & 3) == 0) { // (the same for every thread)
            *(uint32_t *)(aq + r * P + c) = q ^ 0x80808080u;
            continue;
          }
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            aq[r * P + c] = (uint8_t)((q >> (8 * b)) ^ 0x80u);
            if (++c == (uint32_t)K) {
              c = 0;
              ++r;
            }
          }
        }
      }
      if (ANY) {
        const int n = M * K;
        if (tid < (n & 3)) {
          const uint32_t q = quant_one<false, true, FAST>(odd, dq_scale, zpf, recip);
          const uint32_t i = (uint32_t)(nvec * 4 + tid), r = i / (uint32_t)K;
          aq[r * P + (i - r * (uint32_t)K)] = (uint8_t)(q ^ 0x80u);
        }
        // what rounds a row up counts as 0 in the row sums
        const int c = K + (tid & 15);
        if ((tid >> 4) < M && c < P)
          aq[(tid >> 4) * P + c] = 0;
      }
    };
    if (scale_is_tame(dq_scale)) // the same for every thread
      quantize(std::true_type{});
    else
      quantize(std::false_type{});
    lds_barrier();
  }

  typedef int vacc __attribute__((ext_vector_type(REGS)));
  vacc acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < REGS; ++r)
        acc[t][c][r] = 0;
  const bool need_rs = ep.need_rowsum;
  int32_t rsp[RT]; // this lane's share of rowsum(A') of row t*T + lane % T
#pragma unroll
  for (int t = 0; t < RT; ++t)
    rsp[t] = 0;
  const v4i flip = {(int)0x80808080, (int)0x80808080, (int)0x80808080,
      (int)0x80808080};
  const v4i zero = {0, 0, 0, 0};

  // RS: row sums of A are needed, fixed outside the loop so that its body has no
  // branch.
  auto consume = [&](int kt, Batch &t, auto RS) {
    v4i a[RT][U][SUBS];
    if (STG) {
      // Through the wave's own piece of LDS into operand order.  The LDS
      // instructions of a wave execute in order; the fences keep the compiler
      // from moving the reads above the writes of other lanes, and the next
      // batch's writes above these reads.
      uint8_t *const stg = lds_raw + wave * kStageWave;
      // (the same for the whole wave)
      if (ANY && ((kt + U) * BK > K || kt + U > kt_end)) {
        const int s = kt + (lane % CPR) / 4;
        const int k0 = s * BK + (lane & 3) * 16;
        constexpr uint64_t kFill = A_MODE == 1 ? 0x8080808080808080ull : 0;
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
          const int row = j * RPI + lane / CPR;
          const int left = s < kt_end && row < M ? K - k0 : 0;
          const int len = left < 0 ? 0 : left < 16 ? left : 16;
          // bytes the load was moved back by: < 16 where the chunk has any
          const int back = row * K + k0 - (M * K - 16);
          t.a[j] = row_chunk(t.a[j], back > 0 && len > 0 ? back : 0, len, kFill);
        }
      }
#pragma unroll
      for (int j = 0; j < NLD; ++j)
        *(v4i *)(stg + (j * RPI + lane / CPR) * kPitch + (lane % CPR) * 16) =
            A_MODE == 1 ? t.a[j] ^ flip : t.a[j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int b = 0; b < SUBS; ++b)
            a[r][u][b] = *(const v4i *)(stg + (r * T + lr) * kPitch +
                                        (u * 4 + b * 2 + lk) * 16);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k0 = (kt + u) * BK + lk * 16;
        const bool in = kt + u < kt_end && k0 < K;
        if (DQ) {
#pragma unroll
          for (int r = 0; r < RT; ++r) {
            const int row = r * 16 + lr;
            a[r][u][0] = *(const v4i *)(aq + (row < M ? row : 0) * P + (in ? k0 : 0));
            if (decltype(RS)::value)
              a[r][u][0] = in ? a[r][u][0] : zero;
          }
        } else {
          a[0][u][0] = A_MODE == 1 ? t.a[u] ^ flip : t.a[u];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < RT; ++r) {
#pragma unroll
        for (int b = 0; b < SUBS; ++b) {
          if (decltype(RS)::value)
            rsp[r] += frag_rowsum(a[r][u][b]);
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            if constexpr (T == 32)
              acc[r][c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                  a[r][u][b], t.b[u][c][b], acc[r][c], 0, 0, 0);
            else
              acc[r][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                  a[r][u][b], t.b[u][c][b], acc[r][c], 0, 0, 0);
          }
        }
      }
  };
  auto k_loop = [&](auto RS) {
    int kt = kt_begin;
    if (DQ) {
      consume(kt, first, RS);
      kt += U;
    }
    for (; kt < kt_end; kt += U) {
      Batch t;
      request(kt, t);
      consume(kt, t, RS);
    }
  };
  if (need_rs)
    k_loop(std::true_type{});
  else
    k_loop(std::false_type{});
  if (A_MODE == 1 && need_rs && !ANY) {
    // A chunk outside the slice or past K was read as zeros, that is 16 times
    // -128 behind the flip: taken out of the row sums again.  Those are the
    // steps that fill the last batch up, and chunks of the very last step of K.
    // (Counted, not looked for step by step: 4 rows, K=11008 N=4608 13.9 -> 11.9
    // us, 24 rows 14.8 -> 13.1.)
    const int steps = kt_end - kt_begin;
    int out = (U - 1 - (steps + U - 1) % U) * SUBS;
    if (steps > 0 && kt_end == KT)
#pragma unroll
      for (int b = 0; b < SUBS; ++b)
        out += (KT - 1) * BK + (b * 2 + lk) * 16 >= K;
#pragma unroll
    for (int t = 0; t < RT; ++t)
      rsp[t] += out * 2048;
  }
  __syncthreads(); // every wave is done reading its rows from LDS

  // Accumulator layout: lane holds column lane % T; register r holds row
  // 4*(lane/16) + r of a 16x16 tile, 8*(r/4) + 4*(lane/32) + r%4 of a 32x32 one.
  // Slot (tile, r) is finished by wave slot % 8.
#pragma unroll
  for (int t = 0; t < RT; ++t) {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < REGS; ++r)
        part[wave][(t * CT + c) * REGS + r][lane] = acc[t][c][r];
    if (need_rs) {
      int32_t rs = rsp[t];
#pragma unroll
      for (int off = T; off < 64; off *= 2)
        rs += __shfl_xor(rs, off, 64);
      if (lane < T)
        atomicAdd(&rowsum[t * T + lane], rs);
    }
  }
  __syncthreads();
  if (!col_ok)
    return;
  const int32_t db = ob - (has_bzp ? bz : 0);
  const float bj = has_bias ? bias : -0.0f;
  float sj = 0.0f;
  if (EPI != kEpiI32) {
    sj = (DQ ? dq_scale : as) * bs;
    if (EPI == kEpiQ8)
      sj = sj / ys;
  }
#pragma unroll
  for (int h = 0; h < (SLOTS + WAVES - 1) / WAVES; ++h) {
    const int e = h * WAVES + wave;
    const int rt = e / REGS / CT, r = e % REGS;
    const int row = T == 32 ? 8 * (r >> 2) + 4 * lk + (r & 3) : 4 * lk + r;
    const int m = rt * T + row;
    if (e >= SLOTS || m >= M)
      continue;
    uint32_t y = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      y += (uint32_t)part[w][e][lane];
    int32_t da = oa - (DQ ? dq_zp : has_azp ? az : 0);
    if (!DQ && ep.a_zp_len > 1)
      da = oa - load_zp_i32(ep.a_zp, A_OFF, m);
    y += (uint32_t)da * (uint32_t)cs;
    if (need_rs)
      y += (uint32_t)db * (uint32_t)rowsum[m];
    y += (uint32_t)K * (uint32_t)da * (uint32_t)db;
    store_one<EPI>(ep, (int64_t)m * N + n, y, sj, yz, bj);
  }
}

// Rows that only the ANY form takes.
bool any_rows(const GemmArgs &g) {
  return g.K % 16 != 0 || (!g.X && (((uintptr_t)g.A) & 15) != 0);
}

template <int A_MODE, int EPI, int DQ, int T, int RT, int CT, bool STG>
void launch_one(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  note_gemm_kernel(
      DQ ? (CT == 2 ? "k_gemm_i8_skinny (rows quantized in the kernel, 2 x 16 columns)"
                    : "k_gemm_i8_skinny (rows quantized in the kernel, 16 columns)")
      : T == 32 ? "k_gemm_i8_skinny (32 columns)"
      : CT == 2 ? "k_gemm_i8_skinny (2 x 16 columns)"
      : STG     ? "k_gemm_i8_skinny (16 columns)"
                : "k_gemm_i8_skinny (16 columns, rows loaded directly)");
  auto *kernel = k_gemm_i8_skinny<A_MODE, EPI, DQ, T, RT, CT, STG, false>;
  if constexpr (DQ || STG)
    if (any_rows(g))
      kernel = k_gemm_i8_skinny<A_MODE, EPI, DQ, T, RT, CT, STG, true>;
  kernel<<<(unsigned)((g.N + T * CT - 1) / (T * CT)), WAVES * 64, 0, st>>>(
      SkinnyArgs{DQ ? (const void *)g.X : g.A, g.Bp, (int)g.M, (int)g.N, (int)g.K,
          pack_epi(ep, EPI)});
}
// Blocks of 16 columns are what fills the device while N / 16 is up to 256.
constexpr int64_t kOneRound = 256 * 16;

// One column tile of 16 per block, or two.  Beyond one round of blocks one is
// still ahead where a block does little besides streaming weights (1 row it
// quantizes, K=4096 N=4608: 4.6 / 5.2 us, N=11008: 6.6 / 7.1), and two where its own
// work is large against them: K is short (1 row, K=1024 N=11008: 5.2 / 4.8 us; 5
// rows it quantizes, K=2048 N=5120: 5.1 / 4.4, K=2688 N=11008: 7.3 / 6.9), or it
// quantizes more than 16 Ki elements of more than four rows (8 rows of 4096,
// N=6144: 8.2 / 7.4, N=11008: 13.5 / 10.1; but 4 rows of 8192, N=6144: 12.1 / 13.6).
template <int A_MODE, int EPI, int DQ, int RT, bool STG>
void launch_16(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  const bool two = DQ ? g.K <= 3072 || (g.M > 4 && g.M * g.K > 16384)
                      : g.K <= 1024;
  if (g.N > kOneRound && two)
    launch_one<A_MODE, EPI, DQ, 16, RT, 2, STG>(st, g, ep);
  else
    launch_one<A_MODE, EPI, DQ, 16, RT, 1, STG>(st, g, ep);
}

template <int A_MODE, int EPI>
void launch_rows(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  const bool rounds = g.N > kOneRound;
  if (g.M <= 4) {
    // Rows loaded directly, with four steps of weights on their way, up to one
    // round of blocks and for short K (4 rows, K=8192 N=4096: 4.9 us against 5.9
    // through LDS, K=1536 N=11008 4.1 / 4.2); beyond, other blocks' waves hide the
    // loads better (K=11008 N=5120: 12.1 / 9.9, K=2688 N=7808: 4.6 / 4.0).
    if (any_rows(g))
      launch_16<A_MODE, EPI, 0, 1, true>(st, g, ep);
    else if (!rounds || g.K <= 2048)
      launch_16<A_MODE, EPI, 0, 1, false>(st, g, ep);
    else
      launch_one<A_MODE, EPI, 0, 16, 1, 1, true>(st, g, ep);
  } else if (g.M <= 16) {
    launch_16<A_MODE, EPI, 0, 1, true>(st, g, ep);
  } else if (g.M <= 32) {
    // Beyond one round one 32 x 32 tile beats two of 16 x 16 (24 rows, K=2688
    // N=5120: 4.9 / 3.9 us, K=11008 N=4608: 13.1 / 12.0), unless the column tiles
    // lie a multiple of 128 KiB apart: as many streams at one distance hit the
    // same channels (K=8192 N=4608: 9.7 / 11.0).
    if (rounds && g.K % 4096 != 0)
      launch_one<A_MODE, EPI, 0, 32, 1, 1, true>(st, g, ep);
    else
      launch_one<A_MODE, EPI, 0, 16, 2, 1, true>(st, g, ep);
  } else if (rounds) {
    // more than 32 rows beyond one round: one 32-column tile (64 rows, K=4096
    // N=6144: 16.0 us with 16 columns, 13.2 so; N=4096: 12.7 / 13.1)
    launch_one<A_MODE, EPI, 0, 32, 2, 1, true>(st, g, ep);
  } else if (g.M <= 48) {
    launch_one<A_MODE, EPI, 0, 16, 3, 1, true>(st, g, ep);
  } else {
    launch_one<A_MODE, EPI, 0, 16, 4, 1, true>(st, g, ep);
  }
}

template <int A_MODE>
void launch_epi(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  if (g.epi == kEpiI32)
    launch_rows<A_MODE, kEpiI32>(st, g, ep);
  else if (g.epi == kEpiF32)
    launch_rows<A_MODE, kEpiF32>(st, g, ep);
  else
    launch_rows<A_MODE, kEpiQ8>(st, g, ep);
}

} // namespace

// Whether the kernel can quantize this activation itself (DQ).
bool skinny_quantizes_rows(int64_t M, int64_t K, const void *x) {
  return M >= 1 && M <= 32 && K > 0 && K <= kSkinnyDqBytes &&
         M * round_up(K, 16) <= kSkinnyDqBytes && ((((uintptr_t)x) & 15) == 0);
}

// (K: the offsets of 64 rows and of a column tile's operands stay in 31 bits.)
bool skinny_ok(int64_t M, int64_t K) {
  return M >= 1 && M <= 64 && K > 0 && K < (1 << 24) && M * K >= 16;
}

hipError_t launch_gemm_skinny(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode) {
  if (g.X) {
    if (g.epi != kEpiF32 || !skinny_quantizes_rows(g.M, g.K, g.X))
      return hipErrorInvalidValue;
    const int64_t elements = g.M * g.K;
    // As few float4 per thread as the rows need: 32 x 256, N=3072 in the form for
    // 32 Ki elements 5.1 us against 4.4.
    auto launch_dq = [&](auto rt) {
      constexpr int RT = decltype(rt)::value;
      if (elements <= 4 * 4 * 512)
        launch_16<2, kEpiF32, 4, RT, false>(st, g, ep);
      else if (elements <= 8 * 4 * 512)
        launch_16<2, kEpiF32, 8, RT, false>(st, g, ep);
      else
        launch_16<2, kEpiF32, 16, RT, false>(st, g, ep);
    };
    if (g.M > 16)
      launch_dq(std::integral_constant<int, 2>{});
    else
      launch_dq(std::integral_constant<int, 1>{});
    return hipGetLastError();
  }
  if (!skinny_ok(g.M, g.K))
    return hipErrorInvalidValue;
  if (a_mode == 0)
    launch_epi<0>(st, g, ep);
  else if (a_mode == 1)
    launch_epi<1>(st, g, ep);
  else
    launch_epi<2>(st, g, ep);
  return hipGetLastError();
}

} // namespace gemm
} // namespace om
