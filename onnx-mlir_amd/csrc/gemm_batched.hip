// int8 products of two activations, batched (the attention products of a
// transformer: scores Q K^T and context P V over batch x heads), in one launch
// and without a packed copy of the right-hand side.
//
// What is computed is what gemm_kernels.hip computes,
//     Y[i,j] = sum_k (A[i,k] - az[i]) * (B[k,j] - bz[j])        (mod 2^32)
// as sum A'B' + db*rowsum(A') + da*colsum(B') + K*da*db, once per batch entry.
//
// k_gemm_i8_batched
//   Bound: the int32 results (32 x 12 heads of 128x64x128: 25 MB out, 6 MB in;
//   4.5 us at the 5.66 TB/s the device stores at) and, with one K step, the
//   chain load -> LDS -> MFMA -> store of a block.  Measured 6.1 us = 5.1 TB/s.
//   Why one launch: packing B and multiplying, matrix by matrix, is three
//   launches of 1.3 to 3.5 us an entry, whatever the entry's size (the same
//   product: 3.5 ms).
//   Why B is transposed here: it is used by M / 64 blocks and never again, so
//   an operand-order copy in memory costs more than it saves.  A thread reads
//   4 columns x 4 or 8 rows of B as 4-byte words (a wave: whole rows of the
//   tile), turns 4 x 4 byte blocks around with eight v_perm_b32, and writes the
//   columns' K bytes into LDS in operand order; column sums are two dot
//   products of registers it holds anyway.
//   Why 64 x 128 (64 x 64 for N <= 64): 384 entries of 128 x 128 are 768
//   blocks, three per CU, so that one block's stores run beside another's
//   loads.
//   LDS layout of B: [column tile of 32][16-byte K chunk][column][16 bytes],
//   the column's place within its group of four XORed with (column / 16) % 4:
//   the 4- and 8-byte writes of a wave (columns four apart) and the 16-byte
//   operand reads then both touch every bank equally often.
//   Loads: buffer loads with a lane offset that never changes (64-bit addresses
//   per load: 2 x 256x4096x4096 50.4 us, this form 38.4), two K steps in
//   flight; results written through where row pieces are whole lines (8.6 ->
//   7.5 us, streaming stores 7.9).  Four blocks a CU where 128 registers suffice
//   (96 x 512x64x512 22.6 -> 20.3 us against three), three for the 128-wide
//   unaligned form (four, with 19 spilled: 88 x 472x472x128 15.9 us, three 13.2).
//   Rows at any address: one 32-bit offset and one minimum a load; shifts and
//   masks only in the steps that the end of K lies in (with them, and 64-bit
//   addresses, in every load: 88 x 472x472x128 19.0 us, so 13.2; 56 x 293x293x80 11.8
//   / 8.7; 64 x 511x511x64 13.5 / 9.2; aligned rows 88 x 480x480x128 12.4 / 11.5).
#include "gemm_batched_out.h"
#include "gemm_common.h"
#include "gemm_epilogue.h"

namespace om {

using namespace gemm;

namespace {

constexpr int BM = 64;
constexpr int kBatchDims = GemmBatch::kDims;

struct BatchParams {
  const uint8_t *A, *B;
  int64_t a_total, b_total; // bytes behind A and B
  int M, N, K;
  uint32_t a_flip, b_flip; // 0x80808080 for uint8 operands
  int tiles_m, tiles_n;
  int first;       // batch entry of the launch's first block
  unsigned blocks; // of the launch
  int dims[kBatchDims];    // sizes of the batch dimensions, outermost first
  int64_t a_step[kBatchDims], b_step[kBatchDims]; // in matrices; 0 broadcasts
  bool a_zp_per_matrix, b_zp_per_matrix;
};
// The usual batch, one dimension that A and B step through or share a matrix of
// (the runtime merges dimensions where it can), in 40 bytes: with PackedEpi, whose
// colsum holds B, the arguments are cheap to launch with (from C, 84 x 8x32x8 4.4 -> 3.2
// us a call, 48 x 38x38x80 4.9 -> 3.7, 264 x 31x31x128 5.1 -> 4.1).
struct FlatBatch {
  const uint8_t *A;
  int M, N, K;
  int first;
  unsigned blocks, a_mats, b_mats;
  unsigned a_unsigned : 1, a_steps : 1, b_steps : 1, a_zp_per_matrix : 1,
      b_zp_per_matrix : 1;
};
static_assert(cheap_arguments(sizeof(FlatBatch) + sizeof(PackedEpi), 0));
__device__ __forceinline__ BatchParams expand(const FlatBatch &f, const PackedEpi &p,
    int bn) {
  BatchParams b = {};
  b.A = f.A;
  b.B = (const uint8_t *)p.colsum;
  b.a_total = (int64_t)f.M * f.K * f.a_mats;
  b.b_total = (int64_t)f.K * f.N * f.b_mats;
  b.M = f.M;
  b.N = f.N;
  b.K = f.K;
  b.a_flip = f.a_unsigned ? 0x80808080u : 0u;
  b.b_flip = p.b_unsigned ? 0x80808080u : 0u;
  b.tiles_m = (f.M + BM - 1) / BM;
  b.tiles_n = bn == 64 ? 1 : (f.N + bn - 1) / bn;
  b.first = f.first;
  b.blocks = f.blocks;
  for (int d = 0; d < kBatchDims; ++d)
    b.dims[d] = 1; // (of the first nothing is asked)
  b.a_step[0] = f.a_steps;
  b.b_step[0] = f.b_steps;
  b.a_zp_per_matrix = f.a_zp_per_matrix;
  b.b_zp_per_matrix = f.b_zp_per_matrix;
  return b;
}

// Results leave the matrix cores as 32 columns by two rows to a store: whole lines
// only where rows are multiples of 128 bytes.  Otherwise, by the rule of out_form, a
// block puts its tile into LDS, byte o of what goes to `to` at byte (to & 15) + o, and
// writes it from there in aligned pieces of 16 bytes, written through like whole lines
// are.
//
// `bytes` bytes of int32 results that lie one after the other (a tile as wide as the
// matrix), `to` a multiple of 4.
__device__ __forceinline__ void tile_out(const uint8_t *lds, char *to, int bytes) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const TilePieces p = tile_pieces((int)(uintptr_t)to & 15, bytes);
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(to - p.skew, 0, p.end, 0x00020000);
  const int tid = (int)threadIdx.x;
  for (int o = p.first + tid * 16; o < p.last; o += 256 * 16)
    __builtin_amdgcn_raw_buffer_store_b128(
        *(const u4 *)(lds + o), rsrc, o, 0, kAuxThrough);
  const int o = tile_end(p, tid);
  if (o >= 0)
    __builtin_amdgcn_raw_buffer_store_b32(*(const int *)(lds + o), rsrc, o, 0, 0);
}
// BM rows of BN 4-byte results, kRowPitch bytes apart in LDS, that are whole pieces:
// `tile` and `pitch` are multiples of 16 bytes, and so are `bytes`, those of a row
// that are there.
template <int BN>
constexpr int kRowPitch = BN * 4 + 32;
template <int BN>
__device__ __forceinline__ void rows_out(
    const uint8_t *lds, char *tile, int rows, int bytes, int pitch) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  constexpr int PER = BN / 4, AT_ONCE = 256 / PER; // threads of a row; rows
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      tile, 0, (rows - 1) * pitch + bytes, 0x00020000);
  const int o = (int)threadIdx.x % PER * 16;
#pragma unroll
  for (int q0 = 0; q0 < BM; q0 += AT_ONCE) {
    const int q = q0 + (int)threadIdx.x / PER;
    __builtin_amdgcn_raw_buffer_store_b128(
        *(const u4 *)(lds + q * kRowPitch<BN> + o), rsrc,
        o < bytes ? q * pitch + o : 0x7FFFFFFF, 0, kAuxThrough);
  }
}

// ALIGNED: K % 16 == 0 with A on a 16-byte boundary and N % 4 == 0 with B on a
// 4-byte one, so that every load is whole and inside its row.
// OUT: how results leave, chosen by out_form (gemm_batched_out.h).
template <int BN, int EPI, bool ALIGNED, int OUT>
__device__ __forceinline__ void batched_tile(
    const BatchParams &bp, const EpiParams &ep) {
  static_assert(BN == 128 || BN == 64, "tile width");
  constexpr int TM = BN == 128 ? 2 : 1; // row tiles of 32 per wave
  constexpr int KPT = BN / 16;          // K rows of B per thread
  constexpr int CG = BN / 4;            // groups of four columns
  // The operands of two steps; at the end, results on their way out.
  constexpr int ES = EPI == kEpiQ8 ? 1 : 4;
  constexpr int kOperands = 2 * (BM + BN) * BK;
  constexpr int kStaged = OUT == kOutDirect ? 0 : BM * kRowPitch<BN>;
  static_assert(OUT == kOutDirect || EPI == kEpiI32, "results by way of LDS");
  __shared__ __attribute__((aligned(16)))
  uint8_t sm[kOperands > kStaged ? kOperands : kStaged];
  uint8_t(*const sA)[BM * BK] = (uint8_t(*)[BM * BK])sm;
  uint8_t(*const sB)[BN * BK] = (uint8_t(*)[BN * BK])(sm + 2 * BM * BK);
  __shared__ int32_t s_rowsum[BM], s_da[BM];
  __shared__ int32_t s_colsum[BN];

  // The tiles of one batch entry go to one XCD, whose L2 then holds its A and B.
  int pid = blockIdx.x;
  {
    const int per = (int)bp.blocks >> 3;
    if (per > 0 && pid < per * 8)
      pid = (pid & 7) * per + (pid >> 3);
  }
  const int M = bp.M, N = bp.N, K = bp.K;
  const int tiles = bp.tiles_m * bp.tiles_n;
  const int rank = pid / tiles; // among the launch's entries
  const int entry = bp.first + rank;
  const int t = pid - rank * tiles;
  const int tm = t / bp.tiles_n;
  const int m0 = tm * BM, n0 = (t - tm * bp.tiles_n) * BN;
  int64_t ai = 0, bi = 0;
  {
    int rest = entry;
#pragma unroll
    for (int d = kBatchDims - 1; d > 0; --d) {
      const int q = rest / bp.dims[d];
      const int c = rest - q * bp.dims[d];
      rest = q;
      ai += c * bp.a_step[d];
      bi += c * bp.b_step[d];
    }
    ai += rest * bp.a_step[0];
    bi += rest * bp.b_step[0];
  }
  // The entry's matrices, addressed by 32-bit offsets (gemm_batched_ok).
  const uint8_t *const Ae = bp.A + ai * M * K, *const Be = bp.B + bi * K * N;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;

  // A: row tid / 4 of the tile, 16-byte chunk tid % 4 of the K step.
  const int ar = tid >> 2, ac = tid & 3;
  const bool a_row = m0 + ar < M;
  // B: columns 4 cg .. 4 cg + 3, KPT rows from kg * KPT of the K step.
  const int cg = tid % CG, kg = tid / CG;
  const bool b_col = n0 + cg * 4 < N;

  // ALIGNED: buffer loads, lane offsets that never change and the K step as
  // scalar offset; what lies outside the matrices (rows past M and columns past
  // N are sent there) reads as 0.  The scalar offset itself stays inside: the
  // hardware compares the lane offset with the descriptor's size minus it,
  // unsigned.  Otherwise global loads at byte addresses.
  constexpr int kOutside = 0x7FFFFFFF;
  const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)Ae, 0, M * K, 0x00020000);
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)Be, 0, K * N, 0x00020000);
  const int a_off = (m0 + ar) * K + ac * 16;
  const int b_off = kg * KPT * N + n0 + cg * 4;
  const int a_voff = a_row ? a_off : kOutside;
  int b_voff[KPT];
#pragma unroll
  for (int i = 0; i < KPT; ++i)
    b_voff[i] = b_col ? b_off + i * N : kOutside;
  // Otherwise loads at any address, as 32-bit offsets from a base that lies at most
  // 15 (3) bytes in front of the matrix, none of which may end behind the last
  // matrix: those are moved back to end with it (a_last, b_last).  Bytes of the
  // matrix are among them in the last rows only, of B in the last three (N = 1).
  const int64_t a_left = bp.a_total - ai * M * K - 16, b_left = bp.b_total - bi * K * N - 4;
  const int a_back = a_left < 0 ? (int)-a_left : 0, b_back = b_left < 0 ? (int)-b_left : 0;
  typedef const __attribute__((address_space(1))) uint8_t *glb; // (not flat loads)
  const glb a_base = (glb)scalar_ptr(Ae - a_back), b_base = (glb)scalar_ptr(Be - b_back);
  const int a_last = a_left < kOutside ? (int)a_left + a_back : kOutside;
  const int b_last = b_left < kOutside ? (int)b_left + b_back : kOutside;
  const int a_any = (a_row ? a_off : ac * 16) + a_back, b_any = b_off + b_back;

  int32_t rs = 0, cs[4] = {0, 0, 0, 0};
  // Operands on their way from memory: two K steps, so that a step's loads have
  // the time of two to arrive.
  v4i ra0, ra1;
  uint32_t rb0[KPT], rb1[KPT];
  // (Steps past the end load the first step again, which nobody uses: with no
  // branch around a load its wait is exact.)
  auto load = [&](int step, v4i &ra, uint32_t(&rb)[KPT]) {
    const int k0 = step < K ? step : 0;
    if (ALIGNED) {
      ra = __builtin_amdgcn_raw_buffer_load_b128(arsrc, a_voff, k0, 0);
#pragma unroll
      for (int i = 0; i < KPT; ++i)
        rb[i] = __builtin_amdgcn_raw_buffer_load_b32(
            brsrc, b_voff[i], k0 * N, 0);
    } else {
      typedef const __attribute__((address_space(1))) uint32_t u32_any
          __attribute__((aligned(1)));
      typedef const __attribute__((address_space(1))) v4i_any v4i_glb;
      const int a = a_any + k0;
      ra = *(v4i_glb *)(a_base + lane_offset((uint32_t)(a < a_last ? a : a_last)));
#pragma unroll
      for (int i = 0; i < KPT; ++i) {
        const int b = b_any + (k0 + i) * N;
        rb[i] = *(u32_any *)(b_base +
                                   lane_offset((uint32_t)(b < b_last ? b : b_last)));
      }
    }
  };
  // Registers to LDS, as int8 and in operand order.  In the steps that the last
  // three rows of B or the end of K lie in, what was moved back is shifted into
  // place, and bytes past K become 0 in both operands (rows past M and columns past
  // N are never stored).
  auto store = [&](int k0, int buf, v4i ra, uint32_t(&rb)[KPT]) {
    const v4i flip = {(int)bp.a_flip, (int)bp.a_flip, (int)bp.a_flip, (int)bp.a_flip};
    if (k0 + BK > (ALIGNED ? K : K - 3)) {
      const int left = K - (k0 + ac * 16), a = a_any + k0;
      ra = row_chunk(ra, ALIGNED || a < a_last ? 0 : a - a_last,
          left < 0 ? 0 : left < 16 ? left : 16,
          (uint64_t)bp.a_flip << 32 | bp.a_flip);
#pragma unroll
      for (int i = 0; i < KPT; ++i) {
        const int b = b_any + (k0 + i) * N;
        const uint32_t r = ALIGNED || b < b_last ? rb[i] : rb[i] >> ((b - b_last) * 8 & 31);
        rb[i] = k0 + kg * KPT + i < K ? r : bp.b_flip;
      }
    }
    const v4i v = ra ^ flip;
    rs += frag_rowsum(v);
    *(v4i *)(&sA[buf][lds_off(ar, ac)]) = v;
    uint32_t o[4][KPT / 4];
#pragma unroll
    for (int h = 0; h < KPT / 4; ++h) {
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r[i] = rb[h * 4 + i] ^ bp.b_flip;
      const uint32_t t0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);
      const uint32_t t1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
      const uint32_t t2 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
      const uint32_t t3 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
      o[0][h] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
      o[1][h] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
      o[2][h] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
      o[3][h] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
    }
    const int chunk = (kg * KPT) >> 4, within = (kg * KPT) & 15;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int h = 0; h < KPT / 4; ++h)
        cs[j] = __builtin_amdgcn_sdot4((int)o[j][h], 0x01010101, cs[j], false);
      uint8_t *const dst = &sB[buf][((cg >> 3) * 4 + chunk) * 512 +
                                    ((cg & 7) * 4 + ((j ^ (cg >> 2)) & 3)) * 16 +
                                    within];
      if (KPT == 8)
        *(uint64_t *)dst = o[j][0] | ((uint64_t)o[j][KPT / 4 - 1] << 32);
      else
        *(uint32_t *)dst = o[j][0];
    }
  };

  const int ct = BN == 128 ? wave : wave & 1;     // the wave's column tile
  const int rt = BN == 128 ? 0 : (wave >> 1) * 32; // its first row
  v16i acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      acc[i][r] = 0;
  const int bslot =
      ((l32 & ~3) | ((l32 ^ (ct * 2 + (l32 >> 4))) & 3)) * 16;

  // What the epilogue needs per row and column, requested before the operands.
  if (tid < BN)
    s_colsum[tid] = 0;
  if (tid < BM) {
    const int32_t oa = bp.a_flip ? 128 : 0;
    int32_t az = 0;
    if (ep.a_zp_len > 0) {
      const int m = m0 + tid < M ? m0 + tid : 0;
      az = load_zp_i32(ep.a_zp, bp.a_flip != 0,
          ep.a_zp_len > 1 ? (bp.a_zp_per_matrix ? ai * M : 0) + m : 0);
    }
    s_da[tid] = oa - az;
  }
  const int n = n0 + ct * 32 + l32;
  const int nc = n < N ? n : N - 1;
  int32_t db = bp.b_flip ? 128 : 0;
  if (ep.b_zp_len > 0)
    db -= load_zp_i32(ep.b_zp, bp.b_flip != 0,
        ep.b_zp_len > 1 ? (bp.b_zp_per_matrix ? bi * N : 0) + nc : 0);
  float sj = 0.0f;
  int32_t yz = 0;
  if (EPI == kEpiQ8) {
    // (a_scale * b_scale) / y_scale, in this order
    // (src/Conversion/ONNXToKrnl/Math/QLinearMatMul.cpp:127)
    sj = (ep.a_scale[0] * ep.b_scale[ep.b_scale_len == 1 ? 0 : nc]) /
         ep.y_scale[0];
    yz = load_zp_i32(ep.y_zp, ep.y_unsigned, 0);
  }

  auto multiply = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const v4i b = *(const v4i *)(&sB[buf][(ct * 4 + s * 2 + lh) * 512 + bslot]);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v4i a =
            *(const v4i *)(&sA[buf][lds_off(rt + i * 32 + l32, s * 2 + lh)]);
        acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc[i], 0, 0, 0);
      }
    }
  };
  load(0, ra0, rb0);
  if (K <= BK) { // one step: nothing to overlap
    store(0, 0, ra0, rb0);
    __syncthreads();
    multiply(0);
  } else {
    load(BK, ra1, rb1);
    store(0, 0, ra0, rb0);
    lds_barrier();
    for (int k0 = 0;; k0 += 2 * BK) {
      load(k0 + 2 * BK, ra0, rb0);
      multiply(0);
      if (k0 + BK >= K)
        break;
      store(k0 + BK, 1, ra1, rb1);
      lds_barrier();
      load(k0 + 3 * BK, ra1, rb1);
      multiply(1);
      if (k0 + 2 * BK >= K)
        break;
      store(k0 + 2 * BK, 0, ra0, rb0);
      lds_barrier();
    }
  }

  // Row sums: the four threads of a row.  Column sums: the threads of a column
  // group add theirs up in LDS.
  rs += __shfl_xor(rs, 1, 64);
  rs += __shfl_xor(rs, 2, 64);
  if (ac == 0)
    s_rowsum[ar] = rs;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    atomicAdd(&s_colsum[cg * 4 + j], cs[j]);
  __syncthreads();

  // 32x32 accumulator layout: lane holds column lane % 32; register r holds
  // row 8*(r/4) + 4*(lane/32) + r%4.
  const uint32_t csn = (uint32_t)s_colsum[ct * 32 + l32];
  const int rows = M - m0 < BM ? M - m0 : BM, cols = N - n0 < BN ? N - n0 : BN;
  char *const out = (char *)ep.out +
                    (((int64_t)entry * M + m0) * N + n0) * (int64_t)ES;
  // f(first, result) for every register, `first` the row of the lanes 0 .. 31
  auto results = [&](auto f) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int first = rt + i * 32 + 8 * (r >> 2) + (r & 3);
        const uint32_t da = (uint32_t)s_da[first + 4 * lh];
        const uint32_t y =
            (uint32_t)acc[i][r] + da * csn +
            (uint32_t)db * ((uint32_t)s_rowsum[first + 4 * lh] + (uint32_t)K * da);
        f(first, EPI == kEpiI32 ? y : requantize(ep, y, sj, yz));
      }
    }
  };
  auto put = [&](int at, uint32_t v) { *(uint32_t *)(sm + at) = v; };
  const int col = (ct * 32 + l32) * 4;
  if constexpr (OUT == kOutTile) {
    // (as wide as the matrix: its results lie one after the other)
    const int skew = (int)(uintptr_t)out & 15;
    if (n < N)
      results([&](int first, uint32_t v) {
        put(skew + (first + 4 * lh) * N * 4 + col, v);
      });
    __syncthreads();
    tile_out(sm, out, rows * N * 4);
    return;
  }
  if constexpr (OUT == kOutRows) {
    results([&](int first, uint32_t v) {
      put((first + 4 * lh) * kRowPitch<BN> + col, v);
    });
    __syncthreads();
    rows_out<BN>(sm, out, rows, cols * 4, N * 4);
    return;
  }
  // A descriptor over the tile's rows inside the matrix: stores to rows past M
  // fall outside and are dropped (gemm_batched_ok keeps 64 rows below 2^31
  // bytes).
  if (n >= N)
    return;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      out, 0, (int)(((int64_t)rows * N - n0) * ES), 0x00020000);
  const int voff = ((4 * lh) * N + ct * 32 + l32) * ES;
  auto direct = [&](auto aux) {
    results([&](int first, uint32_t v) {
      if (EPI == kEpiI32)
        __builtin_amdgcn_raw_buffer_store_b32(
            (int)v, rsrc, voff + first * N * ES, 0, decltype(aux)::value);
      else
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)v, rsrc,
            voff + first * N * ES, 0, decltype(aux)::value);
    });
  };
  if (N * ES % 128 == 0)
    direct(std::integral_constant<int, kAuxThrough>{});
  else
    direct(std::integral_constant<int, 0>{});
}

template <int BN, bool ALIGNED>
constexpr int kBlocksPerCu = ALIGNED || BN == 64 ? 4 : 3;
template <int BN, int EPI, bool ALIGNED, int OUT>
__global__ __launch_bounds__(256, (kBlocksPerCu<BN, ALIGNED>)) void k_gemm_i8_batched(
    const BatchParams bp, const EpiParams ep) {
  batched_tile<BN, EPI, ALIGNED, OUT>(bp, ep);
}
template <int BN, int EPI, bool ALIGNED, int OUT>
__global__ __launch_bounds__(256, (kBlocksPerCu<BN, ALIGNED>)) void k_gemm_i8_batched_flat(
    const FlatBatch fb, const PackedEpi pe) {
  batched_tile<BN, EPI, ALIGNED, OUT>(expand(fb, pe, BN), unpack_epi<EPI>(pe));
}

template <int BN, int EPI, bool ALIGNED, int OUT>
void launch_out(hipStream_t s, const BatchParams &bp, const EpiParams &ep,
    const FlatBatch *flat) {
  if (!flat) {
    k_gemm_i8_batched<BN, EPI, ALIGNED, OUT><<<bp.blocks, 256, 0, s>>>(bp, ep);
    return;
  }
  PackedEpi pe = pack_epi(ep, EPI);
  pe.colsum = (const int32_t *)bp.B;
  pe.b_unsigned = bp.b_flip != 0;
  k_gemm_i8_batched_flat<BN, EPI, ALIGNED, OUT><<<bp.blocks, 256, 0, s>>>(*flat, pe);
}
template <int BN, int EPI, bool ALIGNED>
void launch_form(hipStream_t s, const BatchParams &bp, const EpiParams &ep,
    const FlatBatch *flat) {
  const OutForm out = out_form(EPI == kEpiI32, bp.M, bp.N, bp.tiles_m, bp.tiles_n,
      (uint64_t)(uintptr_t)ep.out, bp.blocks);
  if constexpr (EPI == kEpiI32) {
    if (out == kOutTile)
      return launch_out<BN, EPI, ALIGNED, kOutTile>(s, bp, ep, flat);
    if constexpr (BN == 128) // (more than one tile to a row)
      if (out == kOutRows)
        return launch_out<BN, EPI, ALIGNED, kOutRows>(s, bp, ep, flat);
  }
  launch_out<BN, EPI, ALIGNED, kOutDirect>(s, bp, ep, flat);
}

template <int EPI>
hipError_t launch_epi(hipStream_t s, const BatchParams &bp, const EpiParams &ep,
    const FlatBatch *flat, bool aligned) {
  if (bp.N <= 64) {
    if (aligned)
      launch_form<64, EPI, true>(s, bp, ep, flat);
    else
      launch_form<64, EPI, false>(s, bp, ep, flat);
  } else {
    if (aligned)
      launch_form<128, EPI, true>(s, bp, ep, flat);
    else
      launch_form<128, EPI, false>(s, bp, ep, flat);
  }
  return hipGetLastError();
}

constexpr int64_t kMaxBytes = (int64_t)1 << 30; // of one matrix, with a tile's overhang
constexpr int64_t kMaxBlocks = (int64_t)1 << 22; // of one launch

int64_t tiles_of(int64_t M, int64_t N) {
  const int64_t bn = N <= 64 ? 64 : 128;
  return ((M + BM - 1) / BM) * ((N + bn - 1) / bn);
}

} // namespace

bool gemm_batched_ok(const GemmArgs &g, const GemmBatch &b) {
  return g.epi != kEpiF32 && g.M > 0 && g.N > 0 && g.K > 0 &&
         (g.M + BM) * g.K < kMaxBytes && (g.K + 4 * BK) * g.N < kMaxBytes && b.count > 0 && b.count <= INT32_MAX &&
         g.M * g.K * b.a_mats >= 16 && g.K * g.N * b.b_mats >= 4 &&
         g.M < kMaxBytes && g.N < ((int64_t)1 << 23) &&
         tiles_of(g.M, g.N) <= kMaxBlocks;
}

// One launch against packing each matrix of B and multiplying entry by entry,
// both by a cost model in microseconds, fitted to 3600 products (1 to 32 entries,
// 1 to 2048 rows, K 32 to 11008, N 32 to 4096, odd sizes among them) when loads at any
// address and launches took longer.  Of 500 timed both ways with the kernels as they
// are, its choice is more than 4 % behind for 13, all but one of them one to three
// entries (1 x 10x4516x38 27.0 us for 10.6), and 0.9 % in the geometric mean; with 1.15
// for rows at any address, which is what long chains show, 1.6 %.
//   One launch: the chain of a block's K steps, or where there are more blocks
//   than the device holds what the CUs have to do in sum.  It does not split K, so
//   few entries with a long K are a few blocks: 1 x 8192 x 128 70 us against 14
//   packed, 16 x 4096 x 4096 37 / 18, four of 1 x 8192 x 128 71 / 54.
//   Packed: the kernels of launch_gemm, two launches and a pass over each matrix of
//   B in front, and the launches' own time on the host: 384 x 128x64x128 7.1 us /
//   3.5 ms, 8 x 1024x1024x1024 29.0 / 79.1, 2 x 1024x4096x1024 40.4 / 52.5.
// Entries above 2^33 multiply-adds go to the tile kernels (1.5 - 2 POP/s against
// the 0.77 reached here; 4 x 2048x2048x2048 89.5 / 93.7).
bool gemm_batched_pays(const GemmArgs &g, const GemmBatch &b) {
  if (g.M * g.N * g.K > ((int64_t)1 << 33))
    return false;
  const double steps = (double)((g.K + BK - 1) / BK);
  const double out_mb = 4e-6 * (double)(g.M * g.N), b_mb = 1e-6 * (double)(g.K * g.N);
  const double count = (double)b.count, mats = (double)b.b_mats;
  const bool narrow = g.N <= 64, chunks = g.K % 16 == 0;
  const double cus = (double)tiles_of(g.M, g.N) * count / 256;
  const double chain = narrow ? 0.34 : 0.54, share = (narrow ? 0.2 : 0.23) * cus;
  const double one = 2.1 + 0.014 * out_mb * count +
                     steps * (chain > share ? chain : share) *
                         (chunks && g.N % 4 == 0 ? 1.0 : 1.57);
  double gemm;
  if (g.M <= 64 && chunks) {
    gemm = 2.7 + steps * (0.036 + 0.0009 * (double)g.M) + 0.088 * b_mb;
  } else if (g.K <= 1024 && g.K % 256 == 0 && g.M * g.N <= ((int64_t)1 << 21)) {
    gemm = 2.4 + 0.06 * steps;
  } else {
    const double tiles = (double)(((g.M + 127) / 128) * ((g.N + 127) / 128)) / 400;
    gemm = 2.7 + (chunks ? 0.28 : 0.7) * steps * (tiles > 1 ? tiles : 1) + 0.12 * out_mb;
  }
  const double device = mats * (3.5 + 0.44 * b_mb) + count * gemm;
  const double host = 2.5 * (2 * mats + count);
  return one <= (device > host ? device : host);
}

hipError_t launch_gemm_batched(
    hipStream_t s, const GemmArgs &g, const GemmBatch &b) {
  if (!gemm_batched_ok(g, b))
    return hipErrorInvalidValue;
  BatchParams bp = {};
  bp.A = (const uint8_t *)g.A;
  bp.B = (const uint8_t *)b.B;
  bp.a_total = g.M * g.K * b.a_mats;
  bp.b_total = g.K * g.N * b.b_mats;
  bp.M = (int)g.M;
  bp.N = (int)g.N;
  bp.K = (int)g.K;
  bp.a_flip = g.a_unsigned ? 0x80808080u : 0u;
  bp.b_flip = g.b_unsigned ? 0x80808080u : 0u;
  bp.tiles_m = (int)((g.M + BM - 1) / BM);
  bp.tiles_n = (int)(tiles_of(g.M, g.N) / bp.tiles_m);
  for (int d = 0; d < kBatchDims; ++d) {
    bp.dims[d] = (int)b.dims[d];
    bp.a_step[d] = b.a_step[d];
    bp.b_step[d] = b.b_step[d];
  }
  bp.a_zp_per_matrix = b.a_zp_per_matrix;
  bp.b_zp_per_matrix = b.b_zp_per_matrix;
  EpiParams ep = {};
  ep.a_zp = g.a_zp;
  ep.a_zp_len = g.a_zp ? g.a_zp_len : 0;
  ep.b_zp = g.b_zp;
  ep.b_zp_len = g.b_zp ? g.b_zp_len : 0;
  ep.a_scale = g.a_scale;
  ep.b_scale = g.b_scale;
  ep.b_scale_len = g.b_scale_len;
  ep.y_scale = g.y_scale;
  ep.y_zp = g.y_zp;
  ep.out = g.out;
  ep.y_unsigned = g.y_unsigned;
  ep.narrow = (int)g.narrow;
  const bool aligned = g.K % 16 == 0 && g.N % 4 == 0 &&
                       (((uintptr_t)g.A) & 15) == 0 && (((uintptr_t)b.B) & 3) == 0;
  note_gemm_kernel("k_gemm_i8_batched");
  const int last = kBatchDims - 1; // (one dimension: the others are 1)
  const bool one = b.count == b.dims[last] && b.a_step[last] <= 1 &&
                   b.b_step[last] <= 1 && b.a_mats <= INT32_MAX &&
                   b.b_mats <= INT32_MAX;
  FlatBatch fb = {};
  fb.A = bp.A;
  fb.M = bp.M;
  fb.N = bp.N;
  fb.K = bp.K;
  fb.a_mats = (unsigned)b.a_mats;
  fb.b_mats = (unsigned)b.b_mats;
  fb.a_unsigned = g.a_unsigned;
  fb.a_steps = b.a_step[last] != 0;
  fb.b_steps = b.b_step[last] != 0;
  fb.a_zp_per_matrix = b.a_zp_per_matrix;
  fb.b_zp_per_matrix = b.b_zp_per_matrix;
  const int64_t per_launch = kMaxBlocks / tiles_of(g.M, g.N);
  for (int64_t e = 0; e < b.count; e += per_launch) {
    const int64_t entries = b.count - e < per_launch ? b.count - e : per_launch;
    bp.first = (int)e;
    bp.blocks = (unsigned)(entries * bp.tiles_m * bp.tiles_n);
    fb.first = bp.first;
    fb.blocks = bp.blocks;
    const FlatBatch *const flat = one ? &fb : nullptr;
    const hipError_t rc = g.epi == kEpiI32 ? launch_epi<kEpiI32>(s, bp, ep, flat, aligned)
                                           : launch_epi<kEpiQ8>(s, bp, ep, flat, aligned);
    if (rc != hipSuccess)
      return rc;
  }
  return hipSuccess;
}

} // namespace om
