// int8 GEMM for gfx950 on the matrix cores (v_mfma_i32_32x32x32_i8), with the
// zero-point correction applied exactly in int32 and the epilogues of
// MatMulInteger (int32), MatMulInteger+Cast+Mul (f32) and QLinearMatMul
// (8-bit requantize) fused into the store.
//
// What is computed (src/Conversion/ONNXToKrnl/Math/MatMulInteger.cpp:59-90,
// src/Conversion/ONNXToKrnl/Math/QLinearMatMul.cpp:88-138):
//     Y[i,j] = sum_k (A[i,k] - az[i]) * (B[k,j] - bz[j])        (mod 2^32)
// The matrix cores multiply signed 8-bit values, so an unsigned operand is
// moved to int8 by subtracting 128 (XOR 0x80): A = A' + oa, B = B' + ob with
// oa, ob in {0, 128}.  With da[i] = oa - az[i] and db[j] = ob - bz[j]
//     Y[i,j] = sum_k A'B' + db[j]*rowsum(A')[i] + da[i]*colsum(B')[j]
//              + K*da[i]*db[j]                                  (mod 2^32)
// which is exact because int32 addition and multiplication wrap.
//
// Layout: A is used as given ([M,K] row-major, K contiguous).  B is packed
// once into Bp, the order in which the matrix cores consume it (k_pack_b):
//   Bp[nt][ks][sub][lane][16 bytes], nt = column / 32, ks = K step of 64
//   bytes, sub = half step; lane l holds, for column nt*32 + l%32, the 16 K
//   bytes starting at ks*64 + (sub*2 + l/32)*16
// int8 (u8 shifted by -128), zero filled up to [Npad, Kpad].  The operand of
// one MFMA is one contiguous KiB, 16 bytes per lane, whether it is loaded
// into registers or copied into LDS.
//
// Kernels (all walk K in steps of 64 bytes):
//   k_gemm_i8_dma        A and Bp tiles copied from global memory straight
//                        into a ring of three LDS stages; K a multiple of 16
//   k_gemm_i8            tiles staged through registers, LDS double buffered:
//                        the general path, any K, any alignment of A
// and, in files of their own, k_gemm_i8_bs and k_gemm_i8_dma_bs (Bp read straight
// into MFMA operand registers, only A through LDS), k_gemm_i8_skinny (M <= 64,
// weight streaming), k_gemm_i8_flight, k_gemm_i8_wreg and k_gemm_i8_batched.
// k_gemm_i8_dma, k_gemm_i8_dma_bs and k_gemm_i8 also multiply parts of K, which
// k_sum_parts adds up, where a product has few tiles and many K steps (split_plan).
// A tiles in LDS have 64-byte rows whose 16-byte chunk index is XOR-swizzled
// with bits 2..3 of the row (bank-conflict free writes and operand reads); Bp
// tiles in LDS keep their global order.

#include <math.h>

#include <algorithm>

#include "gemm_common.h"
#include "gemm_epilogue.h"

#include <stdlib.h>

namespace om {

using namespace gemm;

namespace {

// BM x BN block tile, WGM x WGN waves, each wave a (BM/WGM) x (BN/WGN) tile
// made of 32x32 MFMA tiles.  MINB: blocks that a CU is to hold.  Three of 64 x 128,
// without spilled registers; a fourth, which spills 4 of its 128 registers a lane, is
// 0.3 % slower in the geometric mean of 1002 products (in us, four / three: int32 4099 x
// 777 x 1001 with row sums 15.4 / 13.9, 2717 x 88 x 2204 8.0 / 9.3).
// A_MODE: 0 = int8 as is, 1 = uint8 (XOR 0x80 while staging), 2 = already
// shifted (stored as u8-128) -- offsets as for uint8, no XOR.
// A_LOAD: kLoadAligned = K % 64 == 0 and A 16-byte aligned (plain vector
// loads); kLoadAny = any K and alignment, at least 16 bytes of A (16-byte
// loads at byte addresses, the bytes past the end of a row replaced); kLoadBytes
// = byte loads (an A of fewer than 16 bytes, K = 0).
template <int BM, int BN, int WGM, int WGN, int MINB, int A_MODE, int EPI,
    int A_LOAD, bool SPLIT = false>
__global__ __launch_bounds__(WGM *WGN * 64, MINB) void k_gemm_i8(TileArgs args) {
  const uint8_t *__restrict__ A = args.A;
  const int8_t *__restrict__ Bp = args.Bp;
  const int M = args.M, N = args.N, K = args.K;
  const int Kpad = A_LOAD == kLoadAligned ? K : padded_k(K);
  const int tiles_m = tiles_of(M, BM), tiles_n = tiles_of(N, BN);
  const EpiParams ep = unpack_epi<EPI>(args.epi);
  const KSplit ks = {args.steps, part_stride(M, N)};
  constexpr int THREADS = WGM * WGN * 64;
  constexpr int WTM = BM / WGM, WTN = BN / WGN; // wave tile
  constexpr int TM = WTM / 32, TN = WTN / 32;   // MFMA tiles per wave
  constexpr int CH_A = BM * 4 / THREADS;        // 16-byte chunks per thread
  constexpr int CH_B = BN * 4 / THREADS;
  static_assert(BM * 4 % THREADS == 0 && BN * 4 % THREADS == 0, "tile/threads");

  __shared__ __attribute__((aligned(16))) uint8_t sA[2][BM * BK];
  __shared__ __attribute__((aligned(16))) uint8_t sB[2][BN * BK];

  // Tile order.  Consecutive workgroup ids are dealt round-robin to the 8
  // XCDs, each with its own L2; renumber so that one XCD gets a contiguous
  // range, then walk that range in groups of 8 tile rows so the tiles resident
  // on an XCD share a few A panels and Bp panels.
  int pid = blockIdx.x;
  {
    const int nb = tiles_m * tiles_n;
    const int per = nb >> 3;
    if (per > 0 && pid < per * 8)
      pid = (pid & 7) * per + (pid >> 3);
  }
  constexpr int GROUP = 8;
  const int in_group = GROUP * tiles_n;
  const int group = pid / in_group;
  const int first_m = group * GROUP;
  const int gsize = (tiles_m - first_m < GROUP) ? tiles_m - first_m : GROUP;
  const int tm = first_m + (pid % in_group) % gsize;
  const int tn = (pid % in_group) / gsize;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // wave index as a scalar: everything derived from it (tile origin, LDS
  // bases, output rows) then lives in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;


  constexpr int kFill = (A_MODE == 1) ? (int)0x80808080 : 0;
  const int KTs = Kpad / BK; // K steps: stride between column tiles of Bp

  // kLoadAny: this thread's chunks in K step 0 (rows past M clamped to the
  // last row, as below) and the last address a 16-byte load may have.
  const uint8_t *arow[CH_A];
  const uint8_t *alast = nullptr;
  if (A_LOAD == kLoadAny) {
#pragma unroll
    for (int h = 0; h < CH_A; ++h) {
      const int q = tid + h * THREADS;
      const int gm = m0 + (q >> 2) < M ? m0 + (q >> 2) : M - 1;
      arow[h] = A + (int64_t)gm * K + (q & 3) * 16;
    }
    alast = A + ((int64_t)M * K - 16);
  }

  // Global loads only fetch; uint8 data is shifted to int8 after it is read
  // back from LDS.  In the general paths bytes past the end of a row are
  // replaced by the byte that the shift maps to 0.
  auto load_global = [&](int k0, v4i(&ra)[CH_A], v4i(&rb)[CH_B]) {
#pragma unroll
    for (int h = 0; h < CH_A; ++h) {
      const int q = tid + h * THREADS;
      const int r = q >> 2, c = q & 3;
      const int gm = m0 + r;
      const int gk = k0 + c * 16;
      v4i v = {kFill, kFill, kFill, kFill};
      if (A_LOAD == kLoadAligned) {
        // K % 64 == 0, so every chunk lies inside its row.  Rows past M are
        // clamped to the last row: they only feed output rows that are never
        // stored, and an unconditional load lets the hardware counter of
        // outstanding loads be waited on exactly (a load under a branch
        // would force a full drain).
        const int gmc = gm < M ? gm : M - 1;
        v = *(const v4i *)(A + (int64_t)gmc * K + gk);
      } else if (A_LOAD == kLoadAny) {
        // One 16-byte load per chunk at whatever address the chunk has, moved
        // back to end with the buffer where it would run past it.  What does
        // not belong to the row is taken out when the chunk goes to LDS
        // (mask_tail), one step in K: nothing here waits for the load.  (With
        // the masking here, in every step, each step paid the latency of its
        // own loads: 4099 x 777 x 1001 19.7 us against 16.0, the fused layer
        // 100 x 11000 x 4000 128 against 84.)
        const uint8_t *const p = arow[h] + k0;
        v = *(const v4i_any *)(p < alast ? p : alast);
      } else {
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 16; ++b) {
          const int kk = gk + b;
          uint32_t byte = (uint32_t)kFill & 0xFFu;
          if (gm < M && kk < K)
            byte = A[(int64_t)gm * K + kk];
          w[b >> 2] |= byte << ((b & 3) * 8);
        }
        v = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
      }
      ra[h] = v;
    }
#pragma unroll
    for (int h = 0; h < CH_B; ++h) {
      // Chunk q of the stage's Bp tile: KiB q/64 is (column tile (q/64)/2,
      // half step (q/64)%2), 16 bytes per lane.  Bp is padded to
      // [Npad, Kpad]: always in bounds and aligned.
      const int q = tid + h * THREADS;
      const int ci = q >> 6;
      rb[h] = *(const v4i *)(Bp +
                             ((int64_t)((n0 >> 5) + (ci >> 1)) * KTs +
                                 (k0 >> 6)) * 2048 +
                             (ci & 1) * 1024 + (q & 63) * 16);
    }
  };
  // kLoadAny, the last K step when it is not a whole one: a chunk keeps the
  // K - gk bytes that are the row's, shifted down by as much as its load was
  // moved back; the rest (the next row's, or a whole chunk past the row)
  // becomes the fill byte.  The weights are zero there, but the row sums count
  // what these bytes hold.
  auto mask_tail = [&](v4i(&ra)[CH_A]) {
    const int k0 = Kpad - BK;
#pragma unroll
    for (int h = 0; h < CH_A; ++h) {
      const int gk = k0 + ((tid + h * THREADS) & 3) * 16;
      const int len = K - gk < 0 ? 0 : K - gk < 16 ? K - gk : 16;
      const uint8_t *const p = arow[h] + k0;
      ra[h] = row_chunk(ra[h], p < alast ? 0 : (int)(p - alast), len,
          (uint32_t)kFill | ((uint64_t)(uint32_t)kFill << 32));
    }
  };
  // (`tail`: these are the registers of the last K step and that is not whole)
  auto store_lds = [&](int buf, v4i(&ra)[CH_A], const v4i(&rb)[CH_B], bool tail) {
    if (A_LOAD == kLoadAny && tail)
      mask_tail(ra);
#pragma unroll
    for (int h = 0; h < CH_A; ++h) {
      const int q = tid + h * THREADS;
      *(v4i *)(&sA[buf][lds_off(q >> 2, q & 3)]) = ra[h];
    }
#pragma unroll
    for (int h = 0; h < CH_B; ++h) {
      const int q = tid + h * THREADS;
      *(v4i *)(&sB[buf][q * 16]) = rb[h];
    }
  };

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0;

  const int l32 = lane & 31;
  const int lh = lane >> 5;
  const bool need_rs = ep.need_rowsum;
  int32_t rsp[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    rsp[i] = 0;

  // Operands of half step s (32 of the stage's 64 K bytes) of this wave's tile.
  auto read_frags = [&](int buf, int s2, v4i(&fa)[TM], v4i(&fb)[TN]) {
    const int c = s2 * 2 + lh;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[i] = *(const v4i *)(&sA[buf][lds_off(wm * WTM + i * 32 + l32, c)]);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      fb[j] = *(const v4i *)(&sB[buf][(((wn * TN + j) * 2 + s2) * 64 + lane) *
                                      16]);
  };

  const int kfirst = SPLIT ? (int)blockIdx.y * ks.steps : 0; // in steps
  const int KT = SPLIT && ks.steps < KTs - kfirst ? ks.steps : KTs - kfirst;
  auto kclamp = [&](int step) {
    return (kfirst + (step < KT ? step : KT - 1)) * BK;
  };
  // The block's last step holds the end of the rows and is not a whole one.
  const bool tail =
      A_LOAD == kLoadAny && (K & (BK - 1)) != 0 && kfirst + KT == KTs;
  v4i ra0[CH_A], rb0[CH_B], ra1[CH_A], rb1[CH_B];
  load_global(kclamp(0), ra0, rb0);
  load_global(kclamp(1), ra1, rb1);
  store_lds(0, ra0, rb0, tail && KT == 1);
  load_global(kclamp(2), ra0, rb0);
  lds_barrier();

  // One K step on LDS buffer `buf`: request all operands of the step, put the
  // next step's tile (already in registers) into the other buffer -- every
  // wave finished reading that one before the last barrier --, refill those
  // registers two steps ahead, then run the MFMAs of both half steps.  RS is
  // whether row sums of A are needed, fixed outside the loop so that the loop
  // body has no branch; `stage` is what the step does for those after it.
  auto k_step = [&](int buf, auto RS, auto stage) {
    v4i fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    read_frags(buf, 0, fa0, fb0);
    read_frags(buf, 1, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    stage();
    __builtin_amdgcn_sched_barrier(0);
    const v4i flip = {(int)0x80808080, (int)0x80808080, (int)0x80808080,
        (int)0x80808080};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      // uint8 -> int8 (minus 128) on the operand registers: VALU work that
      // runs beside the MFMAs
      if (A_MODE == 1)
        fa0[i] ^= flip;
      if (decltype(RS)::value)
        rsp[i] += frag_rowsum(fa0[i]);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
            fa0[i], fb0[j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (A_MODE == 1)
        fa1[i] ^= flip;
      if (decltype(RS)::value)
        rsp[i] += frag_rowsum(fa1[i]);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
            fa1[i], fb1[j], acc[i][j], 0, 0, 0);
  };
  // The last two or three steps stand apart: what stages the last tile may have to
  // mask it, and what computes the last one stages nothing.  In the loop every load
  // and LDS store is unconditional (one load past the end is clamped to the last
  // step and its data never consumed), and the loop has one way out, behind an odd
  // step: so the compiler waits for exactly the register set that it is about to
  // store and leaves the other set's loads in flight.  (With a way out between its
  // two steps, the second waited for the loads of the first as well, in us: f32 109 x
  // 10959 x 224 59.0 against 39.6, 320 x 10002 x 3584 54.4 / 39.5, int32 4099 x 777 x 1001
  // with row sums 14.0 / 13.4.  With the mask under a branch in every step, and four
  // blocks of 64 x 128 a CU: 49.0, 45.9, 14.8.)
  auto k_loop = [&](auto RS) {
    auto whole = [&](int buf, int kt, v4i(&ra)[CH_A], v4i(&rb)[CH_B]) {
      k_step(buf, RS, [&] {
        store_lds(buf ^ 1, ra, rb, false);
        load_global(kclamp(kt + 3), ra, rb);
      });
      lds_barrier();
    };
    int kt = 0;
    for (; kt < KT - 3; kt += 2) {
      whole(0, kt, ra1, rb1);
      whole(1, kt + 1, ra0, rb0);
    }
    if (kt == KT - 3) {
      whole(0, kt++, ra1, rb1);
#pragma unroll
      for (int h = 0; h < CH_A; ++h)
        ra1[h] = ra0[h];
#pragma unroll
      for (int h = 0; h < CH_B; ++h)
        rb1[h] = rb0[h];
    }
    if (kt == KT - 2) {
      k_step(kt & 1, RS, [&] { store_lds((kt & 1) ^ 1, ra1, rb1, tail); });
      lds_barrier();
      ++kt;
    }
    k_step(kt & 1, RS, [] {});
  };
  if (need_rs)
    k_loop(std::true_type{});
  else
    k_loop(std::false_type{});
  if constexpr (SPLIT)
    gemm_epilogue<TM, TN, A_MODE, EPI, 0>(acc, rsp, m0 + wm * WTM, n0 + wn * WTN,
        M, N, blockIdx.y == 0 ? K : 0, part_of(ep, ks), blockIdx.y == 0);
  else
    gemm_epilogue<TM, TN, A_MODE, EPI>(
        acc, rsp, m0 + wm * WTM, n0 + wn * WTN, M, N, K, ep);
}

// ---- GEMM, tiles copied from global memory straight into LDS --------------
// gfx950 can write a 16-byte global load into LDS without passing through
// vector registers (global_load_lds_dwordx4): LDS address = M0 + lane * 16, so
// one wave instruction fills 1 KiB of consecutive LDS and the per-lane global
// address decides what lands where.  That removes the register staging, the
// ds_write instructions and the wait that tied them to the loads; a wave only
// issues the copies, waits for its own to land, and meets the others at one
// barrier per K step.
//
// LDS holds a ring of three stages (A tile + Bp tile of one 64-byte K step
// each; the A tile in the XOR-swizzled row layout, the Bp tile as it is in
// global memory).  In step k a wave
//   waits until its copies for step k have landed (those for k+1 stay in
//   flight), passes the barrier -- now every wave's step-k data is in LDS and
//   every wave is done reading stage (k-1)%3 --,
//   issues its copies for step k+2 into stage (k-1)%3,
//   reads the operands of stage k%3 and runs the MFMAs.
// The operand reads are written as inline assembly: the compiler would make
// every LDS read wait for all outstanding copies into LDS, whichever stage
// they target.  The counts waited for below are therefore explicit.
//
// RAGGED: K is a multiple of 16 but not of the K step, 64 (in k_gemm_i8, which
// takes any K, 512 x 784 x 1001 is 11.8 us against 7.4 here).  A form of its own,
// because what its last step takes costs vector operations in every step: whole
// steps through it were 2 to 7 % slower (4096 x 6656 x 768 with 8-bit results 36.4
// us against 38.8, int32 results 1000 x 6656 x 4096 39.8 / 42.6, 4096 x 4096 x 768
// with 8-bit results 24.5 / 25.8).
template <int BN, int NSTAGE, int MINB, int A_MODE, int EPI, bool RAGGED,
    bool SPLIT = false>
__global__ __launch_bounds__(256, MINB) void k_gemm_i8_dma(TileArgs args) {
  // 2 x 2 waves, each a 64 x (BN/2) tile.
  constexpr int BM = 128;
  const uint8_t *__restrict__ A = args.A;
  const int8_t *__restrict__ Bp = args.Bp;
  const int M = args.M, N = args.N, K = args.K, Kpad = padded_k(K);
  const int tiles_m = tiles_of(M, BM), tiles_n = tiles_of(N, BN);
  const EpiParams ep = unpack_epi<EPI>(args.epi);
  const KSplit ks = {args.steps, part_stride(M, N)};
  constexpr int WTM = 64, WTN = BN / 2, TM = 2, TN = WTN / 32;
  static_assert(BN == 128 || BN == 64, "tile width");
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int CB = BN / 64;      // Bp copies per wave and step
  constexpr int CPW = 2 + CB;      // copies per wave and step
  __shared__ __attribute__((aligned(1024))) uint8_t sm[NSTAGE * STAGE];

  int pid = blockIdx.x;
  {
    const int nb = tiles_m * tiles_n;
    const int per = nb >> 3;
    if (per > 0 && pid < per * 8)
      pid = (pid & 7) * per + (pid >> 3);
  }
  constexpr int GROUP = 8;
  const int in_group = GROUP * tiles_n;
  const int group = pid / in_group;
  const int first_m = group * GROUP;
  const int gsize = (tiles_m - first_m < GROUP) ? tiles_m - first_m : GROUP;
  const int tm = first_m + (pid % in_group) % gsize;
  const int tn = (pid % in_group) / gsize;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31;
  const int lh = lane >> 5;

  // Copy addressing.  Copy instruction j of the A tile fills LDS bytes
  // [j*1024, (j+1)*1024): lane -> row j*16 + lane/4, chunk position lane%4,
  // which holds chunk (lane%4) ^ ((row/4)%4) = (lane%4) ^ ((lane/16)%4) of the
  // row.  Copy instruction c of the Bp tile moves KiB c of the stage, which
  // is (column tile c/2, half step c%2), unchanged.  A wave issues copies
  // 2*wave, 2*wave+1 of A and CB consecutive copies of Bp.
  const int KTs = Kpad / BK; // K steps of the operands, and of this block
  const int kfirst = SPLIT ? (int)blockIdx.y * ks.steps : 0;
  const int KT = SPLIT && ks.steps < KTs - kfirst ? ks.steps : KTs - kfirst;
  const int crow = lane >> 2;
  const int cchunk = (lane & 3) ^ ((lane >> 4) & 3);
  // K is a multiple of 16, so a 16-byte chunk lies wholly inside its row or
  // wholly past it.  In a last step that is not whole, the chunks past the row
  // take its last chunk again (klim): the weights are zero there, and the row
  // sums leave them out.
  const int klim = K - 16 - cchunk * 16;
  const uint8_t *ga[2];
  const int8_t *gb[CB];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = (wave * 2 + h) * 16 + crow;
    const int gm = (m0 + r < M) ? m0 + r : M - 1; // rows past M: never stored
    ga[h] = A + (int64_t)gm * K + cchunk * 16;
  }
#pragma unroll
  for (int h = 0; h < CB; ++h) {
    const int c = wave * CB + h;
    gb[h] = Bp + (int64_t)((n0 >> 5) + (c >> 1)) * KTs * 2048 + (c & 1) * 1024 +
            lane * 16;
  }
  typedef __attribute__((address_space(3))) void *lds_ptr;
  typedef const __attribute__((address_space(1))) void *glb_ptr;
  auto copy_step = [&](int k0, int stage) {
    uint8_t *base = sm + stage * STAGE;
    const int ka = !RAGGED || k0 < klim ? k0 : klim;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      __builtin_amdgcn_global_load_lds((glb_ptr)(ga[h] + ka),
          (lds_ptr)(base + (wave * 2 + h) * 1024), 16, 0, 0);
#pragma unroll
    for (int h = 0; h < CB; ++h)
      __builtin_amdgcn_global_load_lds((glb_ptr)(gb[h] + k0 * 32),
          (lds_ptr)(base + BM * BK + (wave * CB + h) * 1024), 16, 0, 0);
  };

  // Operand addressing: sub-step s (0,1) of a stage uses chunk 2*s + lane/32 of
  // row (wave tile row + lane%32); MFMA tile i adds 32 rows = 2048 bytes.
  const unsigned sm_base = (unsigned)(uintptr_t)(lds_ptr)sm;
  unsigned ra[2], rb[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    ra[s] = sm_base + lds_off(wm * WTM + l32, s * 2 + lh);
    rb[s] = sm_base + BM * BK + ((wn * TN * 2 + s) * 64 + lane) * 16;
  }

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0;

  auto kclamp = [&](int step) {
    return (kfirst + (step < KT ? step : KT - 1)) * BK;
  };
#pragma unroll
  for (int p = 0; p < NSTAGE - 1; ++p)
    copy_step(kclamp(p), p);

  // One LDS read of an MFMA operand.  Kept opaque to the compiler, see above;
  // lds_wait<n>() makes the operands it is given valid once at most n reads
  // are still outstanding (reads complete in order).
  auto lds_read = [](v4i &f, unsigned addr, auto off) {
    asm volatile("ds_read_b128 %0, %1 offset:%2"
                 : "=v"(f)
                 : "v"(addr), "n"(decltype(off)::value)
                 : "memory");
  };

  const bool need_rs = ep.need_rowsum;
  int32_t rsp[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    rsp[i] = 0;

  // Weights of a row sum: none for a chunk past the end of the row.
  auto ones = [&](int kt, int s2) {
    return !RAGGED || (kfirst + kt) * BK + (s2 * 2 + lh) * 16 < K ? 0x01010101
                                                                  : 0;
  };

  int stage = 0; // kt % NSTAGE
  // Whether row sums of A are needed is fixed here, outside the loop, so that
  // the loop body has no branch.
  auto k_loop = [&](auto RS) {
    for (int kt = 0; kt < KT; ++kt) {
      const int prev = (stage == 0) ? NSTAGE - 1 : stage - 1;
      // Own copies of step kt have landed; those of the NSTAGE-2 steps after it
      // may still be in flight.
      __builtin_amdgcn_s_waitcnt(0x0F70 | ((NSTAGE - 2) * CPW));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      copy_step(kclamp(kt + NSTAGE - 1), prev);
      __builtin_amdgcn_sched_barrier(0);
      const unsigned soff = (unsigned)(stage * STAGE);
      v4i fa0[TM], fb0[TN], fa1[TM], fb1[TN];
      using O0 = std::integral_constant<int, 0>;
      using O1 = std::integral_constant<int, 2048>;
      lds_read(fa0[0], ra[0] + soff, O0{});
      lds_read(fa0[1], ra[0] + soff, O1{});
      lds_read(fb0[0], rb[0] + soff, O0{});
      if (TN == 2)
        lds_read(fb0[TN - 1], rb[0] + soff, O1{});
      lds_read(fa1[0], ra[1] + soff, O0{});
      lds_read(fa1[1], ra[1] + soff, O1{});
      lds_read(fb1[0], rb[1] + soff, O0{});
      if (TN == 2)
        lds_read(fb1[TN - 1], rb[1] + soff, O1{});
      if (TN == 2)
        asm volatile("s_waitcnt lgkmcnt(4)"
                     : "+v"(fa0[0]), "+v"(fa0[1]), "+v"(fb0[0]), "+v"(fb0[TN - 1])
                     :
                     : "memory");
      else
        asm volatile("s_waitcnt lgkmcnt(3)"
                     : "+v"(fa0[0]), "+v"(fa0[1]), "+v"(fb0[0])
                     :
                     : "memory");
      if (A_MODE == 1) {
  #pragma unroll
        for (int i = 0; i < TM; ++i)
          fa0[i] ^= (v4i){(int)0x80808080, (int)0x80808080, (int)0x80808080,
              (int)0x80808080};
      }
      if (decltype(RS)::value) {
  #pragma unroll
        for (int i = 0; i < TM; ++i)
          rsp[i] += frag_rowsum(fa0[i], ones(kt, 0));
      }
  #pragma unroll
      for (int i = 0; i < TM; ++i)
  #pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
              fa0[i], fb0[j], acc[i][j], 0, 0, 0);
      if (TN == 2)
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(fa1[0]), "+v"(fa1[1]), "+v"(fb1[0]), "+v"(fb1[TN - 1])
                     :
                     : "memory");
      else
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(fa1[0]), "+v"(fa1[1]), "+v"(fb1[0])
                     :
                     : "memory");
      if (A_MODE == 1) {
  #pragma unroll
        for (int i = 0; i < TM; ++i)
          fa1[i] ^= (v4i){(int)0x80808080, (int)0x80808080, (int)0x80808080,
              (int)0x80808080};
      }
      if (decltype(RS)::value) {
  #pragma unroll
        for (int i = 0; i < TM; ++i)
          rsp[i] += frag_rowsum(fa1[i], ones(kt, 1));
      }
  #pragma unroll
      for (int i = 0; i < TM; ++i)
  #pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
              fa1[i], fb1[j], acc[i][j], 0, 0, 0);
      stage = (stage == NSTAGE - 1) ? 0 : stage + 1;
    }
  };
  if (need_rs)
    k_loop(std::true_type{});
  else
    k_loop(std::false_type{});
  // Copies past the last step are still landing in LDS; nothing reads them,
  // but the block must not release its LDS before they are done.
  __builtin_amdgcn_s_waitcnt(0x0F70);

  if constexpr (SPLIT)
    gemm_epilogue<TM, TN, A_MODE, EPI, 0>(acc, rsp, m0 + wm * WTM, n0 + wn * WTN,
        M, N, blockIdx.y == 0 ? K : 0, part_of(ep, ks), blockIdx.y == 0);
  else
    gemm_epilogue<TM, TN, A_MODE, EPI>(
        acc, rsp, m0 + wm * WTM, n0 + wn * WTN, M, N, K, ep);
}

// ---- pack B ---------------------------------------------------------------
// One block transposes a 64(k) x 64(n) tile of B [K,N] through LDS, writes it
// in MFMA operand order (see the top of the file) and adds the tile's column
// sums into colsum with int32 atomics (integer adds commute, so the result
// does not depend on arrival order).
constexpr int PT = 64;

template <bool B_UNSIGNED>
__global__ __launch_bounds__(256) void k_pack_b(const uint8_t *__restrict__ B,
    int64_t K, int64_t N, int KT, int8_t *__restrict__ Bp,
    int32_t *__restrict__ colsum) {
  __shared__ __attribute__((aligned(16))) uint8_t tile[PT][PT + 4];
  const int ks = blockIdx.y; // K step of 64
  const int64_t k0 = (int64_t)ks * PT;
  const int64_t n0 = (int64_t)blockIdx.x * PT;
  const int tid = threadIdx.x;
  // Read: thread -> row k = tid/4, 16 columns starting at (tid%4)*16.
  {
    const int kr = tid >> 2;
    const int nc = (tid & 3) * 16;
    const int64_t k = k0 + kr;
    // Rows that start on 16-byte boundaries (N % 16 == 0, aligned B): one
    // 16-byte load per thread; otherwise, and at the edges, byte by byte.
    const bool rows_aligned = ((N & 15) == 0) && ((((uintptr_t)B) & 15) == 0);
    if (rows_aligned && k < K && n0 + nc + 16 <= N) {
      v4i q = *(const v4i *)(B + k * N + n0 + nc);
      if (B_UNSIGNED)
        q ^= (v4i){(int)0x80808080, (int)0x80808080, (int)0x80808080,
            (int)0x80808080};
      // row stride 68 and nc % 16 == 0: 4-byte aligned
      uint32_t *dst = (uint32_t *)&tile[kr][nc];
      dst[0] = (uint32_t)q.x;
      dst[1] = (uint32_t)q.y;
      dst[2] = (uint32_t)q.z;
      dst[3] = (uint32_t)q.w;
    } else {
#pragma unroll
      for (int b = 0; b < 16; ++b) {
        const int64_t n = n0 + nc + b;
        uint8_t v = B_UNSIGNED ? 0x80 : 0;
        if (k < K && n < N)
          v = B[k * N + n];
        if (B_UNSIGNED)
          v ^= 0x80;
        tile[kr][nc + b] = v;
      }
    }
  }
  __syncthreads();
  // Write: thread -> column n = tid/4, 16-byte chunk c = tid%4 of the step.
  {
    const int nr = tid >> 2;
    const int c = tid & 3;
    uint32_t w[4] = {0, 0, 0, 0};
    int32_t sum = 0;
#pragma unroll
    for (int b = 0; b < 16; ++b) {
      const uint8_t v = tile[c * 16 + b][nr];
      sum += (int32_t)(int8_t)v;
      w[b >> 2] |= (uint32_t)v << ((b & 3) * 8);
    }
    const int64_t n = n0 + nr;
    // The grid covers [Npad, Kpad] exactly: every byte of Bp is written.
    const int64_t o =
        ((((n >> 5) * KT + ks) * 2 + (c >> 1)) * 64 + (c & 1) * 32 + (n & 31)) *
        16;
    *(v4i *)(Bp + o) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    // Fold the four k-chunks of this column (lanes 4n..4n+3) before the atomic.
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if ((tid & 3) == 0 && sum != 0)
      atomicAdd(&colsum[n], sum);
  }
}

// ---- launch ---------------------------------------------------------------

// Kernel / tile configurations.
enum TileCfg : int {
  kT128x128 = 0, // k_gemm_i8: register-staged tiles (and the general path)
  kD128x128 = 1, // k_gemm_i8_dma: tiles copied straight into LDS
  kB128x256 = 2, // k_gemm_i8_bs: Bp straight into registers
  kD128x64 = 3,  // k_gemm_i8_dma with 128 x 64 tiles
  kW128x384 = 4, // k_gemm_i8_wreg: weights in registers, 12 waves of 32 columns
  kFlight = 5,   // k_gemm_i8_flight: one round of blocks, all operands requested at once
  kB64x256 = 6,  // k_gemm_i8_dma_bs, the same with 64 x 256 tiles
  kB64x128 = 7,  // and with 64 x 128 tiles
  kNumCfg = 8
};

// What the time of a product depends on.
struct Sizes {
  int64_t M, N, K;
  bool bytes;   // 8-bit results
  bool rowsums; // B carries an offset
};
Sizes sizes_of(const GemmArgs &g) {
  return {g.M, g.N, g.K, g.epi == kEpiQ8, g.b_unsigned || g.b_zp_len > 0};
}

// Kernel choice for problems with more than 64 rows, K a multiple of 16 and a
// 16-byte aligned A (anything else takes the general path of k_gemm_i8).
// A tile kernel's time on MI355X:
//   base + steps * max(lone, step * rounds) * (1 + rowsum) + block * b   microseconds.
// A chain of K steps takes as long as the CU with the most blocks, `rounds` of
// them, and what a block does beside it (block4, block1, by the size of a result)
// counts b times, partly the rounds and partly the mean (`round`): CUs that are
// done early leave the others the way to memory.  rowsum: where row sums are added
// up.  Fitted to 2921 products of 65 .. 4096 rows, K and N of 64 .. 11008, each
// timed with every kernel, so that the kernel it names takes the least time
// (profiles/tile_kernel_times.csv): 0.4 % above always taking the fastest, in the
// geometric mean (fitted to two thirds of them, 0.5 % on the rest).  The times
// themselves are within 10 %.  With the mean in the K steps as well, and
// coefficients fitted to 150 products of fewer kinds, it was 1.9 %, and 128 x 64
// tiles were taken too often where K is short and N long (int32 3584 x 320 x 9740
// 39.7 us, in 128 x 128 tiles 33.8; 1903 x 304 x 8576 19.9 / 17.3), 128 x 256 ones for K
// up to 1024 (2048 x 768 x 3072 11.7 / 9.9 in 64 x 128).
struct TileCost {
  TileCfg cfg;
  int bm, bn, trip; // K steps are done in whole trips
  double lone, step, rowsum, block4, block1, base, round;
};
constexpr TileCost kTileCosts[] = {
    {kD128x128, 128, 128, 1, 0.018, 0.298, 0.101, 1.989, 2.474, 2.628, 0.012},
    {kD128x64, 128, 64, 1, 0.069, 0.178, 0.294, 1.006, 1.331, 2.407, 0.003},
    {kB128x256, 128, 256, 4, 0.022, 0.444, 0.126, 3.496, 3.226, 4.769, 0.0},
    {kB64x256, 64, 256, 4, 0.009, 0.231, 0.088, 2.381, 2.323, 3.043, 0.346},
    {kB64x128, 64, 128, 4, 0.027, 0.157, 0.165, 0.756, 0.866, 2.684, 0.331},
};
double tile_us(const TileCost &t, const Sizes &p) {
  const int64_t blocks = ((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn);
  const double rounds = (double)((blocks + 255) / 256);
  const double b = std::max(
      1.0, t.round * rounds + (1.0 - t.round) * (double)blocks / 256.0);
  const double steps = (double)(round_up(p.K, kGemmBK * t.trip) / kGemmBK);
  return t.base + steps * std::max(t.lone, t.step * rounds) *
                      (p.rowsums ? 1.0 + t.rowsum : 1.0) +
         (p.bytes ? t.block1 : t.block4) * b;
}
// Its time, too, where wanted.
// Override for tests and tuning: OM_MI355X_GEMM_TILE=<TileCfg value>.
int choose_tile(const Sizes &p, double *us = nullptr) {
  const char *force = getenv("OM_MI355X_GEMM_TILE");
  if (force && force[0]) {
    const int c = atoi(force);
    if (c >= 0 && c < kNumCfg)
      return c;
  }
  int best = kD128x128;
  double least = tile_us(kTileCosts[0], p);
  for (const TileCost &t : kTileCosts) {
    // (128 x 256 tiles: K a multiple of 256, whole trips of its loop, the step
    // counts its times were taken at)
    if (p.K >= (1 << 24) ? t.trip != 1 : t.cfg == kB128x256 && p.K % 256 != 0)
      continue;
    const double u = tile_us(t, p);
    if (u < least) {
      least = u;
      best = t.cfg;
    }
  }
  if (us)
    *us = least;
  return best;
}

bool gemm_fast_path(int64_t M, int64_t K, const void *A) {
  // K == 0 (an empty sum) has no bytes of A to read: only the general path
  // checks every address against K.
  return M > 16 && K > 0 && K % 16 == 0 && ((((uintptr_t)A) & 15) == 0);
}

// Name of the kernel the calling thread's last launch_gemm chose (for tests
// and reports).
thread_local const char *t_last_kernel = "";
// Whether that kernel wrote GemmArgs::y_limits itself (launch_gemm runs the
// reduction over the output when it did not).
thread_local bool t_limits_written = false;

// The sums of `parts` int32 arrays, each `stride` elements (a multiple of 4)
// after the one before, with the epilogue of a product: 4 consecutive elements
// of the result per thread.  Bound by the launch and by reading the arrays,
// which were written a moment ago (at most 256 tiles of 64 KB).
struct SumArgs {
  const int32_t *in;
  int parts;
  unsigned n, N;
  bool vector_out;
  PackedEpi epi;
};
static_assert(cheap_arguments(sizeof(SumArgs), 0));
template <int EPI>
__global__ __launch_bounds__(256) void k_sum_parts(SumArgs args) {
  const int32_t *__restrict__ in = args.in;
  const int parts = args.parts;
  const unsigned n = args.n, N = args.N;
  const int64_t stride = part_stride(1, n);
  const bool vector_out = args.vector_out;
  const EpiParams ep = unpack_epi<EPI>(args.epi);
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const unsigned o = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (o >= n)
    return;
  float sj[4] = {}, bj[4] = {};
  int32_t yz = 0;
  if (EPI != kEpiI32) {
    const float as = ep.a_scale[0];
    const float ys = EPI == kEpiQ8 ? ep.y_scale[0] : 1.0f;
    if (EPI == kEpiQ8)
      yz = load_zp_i32(ep.y_zp, ep.y_unsigned, 0);
    const bool has_bias = EPI == kEpiF32 && ep.bias != nullptr;
    const float *const bias = has_bias ? ep.bias : ep.b_scale; // always readable
    unsigned c = o % N;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sj[e] = as * ep.b_scale[ep.b_scale_len == 1 ? 0 : c];
      if (EPI == kEpiQ8)
        sj[e] = sj[e] / ys;
      const float bv = bias[has_bias && ep.bias_len > 1 ? c : 0];
      bj[e] = has_bias ? bv : -0.0f;
      c = c + 1 == N ? 0 : c + 1;
    }
  }
  // (the elements past n of the last four lie inside their array's stride)
  u4 y = {0, 0, 0, 0};
  int s = 0;
  for (; s + 4 <= parts; s += 4) {
    u4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = *(const u4 *)(in + (int64_t)(s + q) * stride + o);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      y += v[q];
  }
  for (; s < parts; ++s)
    y += *(const u4 *)(in + (int64_t)s * stride + o);
  uint32_t r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (EPI == kEpiI32) {
      r[e] = y[e];
    } else if (EPI == kEpiF32) {
      const float f = relu_f32((float)(int32_t)y[e] * sj[e] + bj[e], ep.floor);
      r[e] = __float_as_uint(ep.gelu ? gelu_f32(f) : f);
    } else {
      r[e] = requantize(ep, y[e], sj[e], yz);
    }
  }
  if (vector_out && o + 4 <= n) {
    if (EPI == kEpiQ8)
      *(uint32_t *)((uint8_t *)ep.out + o) =
          r[0] | (r[1] << 8) | (r[2] << 16) | (r[3] << 24);
    else
      *(u4 *)((uint32_t *)ep.out + o) = (u4){r[0], r[1], r[2], r[3]};
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (o + e < n) {
      if (EPI == kEpiQ8)
        ((uint8_t *)ep.out)[o + e] = (uint8_t)r[e];
      else
        ((uint32_t *)ep.out)[o + e] = r[e];
    }
}

// What bounds a product whose tiles cover a part of the CUs is the chain of its
// K steps, each the time its operands take into one CU: 0.15 us in 64 x 128 tiles
// of k_gemm_i8_dma_bs, 0.17 in 128 x 64 ones of k_gemm_i8_dma, 0.23 in 128 x 128
// ones, 0.28 in k_gemm_i8, a third to a half more with row sums.  Splitting shortens
// the chain and costs the launch of k_sum_parts, 2.5 us, and the arrays' way through
// memory, 2 us per million elements.  Fitted to 2762 timed splits of 393 products
// in two to 32 parts (within 4 %, root mean square, and within 6 % of 2991 of 200
// products since launches take less; those in k_gemm_i8 to 1994 of 510 products,
// within 5 %).  Taken where that comes out
// ahead of one piece in the tile chosen for it; more than one block per CU gains
// nothing.  K of whole steps in any of the three, other K in k_gemm_i8_dma_bs, whose
// steps do not look for the end of the row (int32 301 x 6384 x 1856 15.4 / 13.8 us).
// Measured in one piece / split: 70 x 8192 x 1024 24.5 / 10.2 us, 118 x 10624 x
// 1536 31.3 / 12.8, 100 x 4096 x 4096 14.4 / 12.9, 148 x 2304 x 832 9.3 / 8.4.
// The plan is made once per product (GemmArgs::split), after the tests that turn
// most products away; parts are looked for around the minimum of the model.
struct SplitForm {
  SplitKernel kernel;
  int64_t tiles, trip;
  double us_step, rowsum, us_else; // us_else: beside steps and arrays
};
SplitForm split_form(SplitKernel kernel, int64_t M, int64_t N) {
  const int64_t tm = (M + 127) / 128, t128 = tm * ((N + 127) / 128);
  switch (kernel) {
  case kSplitDma128:
    return {kernel, t128, 1, 0.230, 0.31, 6.37};
  case kSplitDma64:
    return {kernel, tm * ((N + 63) / 64), 1, 0.173, 0.43, 5.81};
  case kSplitBs:
    return {kernel, ((M + 63) / 64) * ((N + 127) / 128), 4, 0.150, 0.33, 5.85};
  default:
    return {kernel, t128, 1, 0.279, 0.52, 6.68};
  }
}
bool split_possible(const Sizes &p, bool any) {
  // (under 24 steps a second launch is within the model's error, unless they
  // are those of k_gemm_i8)
  return (p.K + kGemmBK - 1) / kGemmBK >= (any ? 8 : 24) &&
         ((p.M + 127) / 128) * ((p.N + 127) / 128) <= 128 &&
         p.M * p.N <= ((int64_t)1 << 22) && p.M * p.K >= 16 && p.K < (1 << 24);
}
// The split of the product in this kernel that takes less than `least`, which it
// lowers.
void try_split(SplitKernel kernel, const Sizes &z, GemmSplit &best, double &least) {
  const SplitForm f = split_form(kernel, z.M, z.N);
  const int64_t KT = (z.K + kGemmBK - 1) / kGemmBK;
  const double us_part = 2.02e-6 * (double)(z.M * z.N);
  const double us_step = f.us_step * (z.rowsums ? 1.0 + f.rowsum : 1.0);
  const int64_t most = 256 / f.tiles < KT / 4 ? 256 / f.tiles : KT / 4;
  // steps * us_step + parts * us_part is least where both are equal
  const int64_t around = (int64_t)sqrt((double)KT * us_step / us_part);
  const int64_t low = around - 2 < most - 4 ? around - 2 : most - 4;
  for (int64_t p = low < 2 ? 2 : low; p <= most && p <= around + 3; ++p) {
    const int64_t steps = round_up((KT + p - 1) / p, f.trip);
    const int64_t parts = (KT + steps - 1) / steps; // (none without a step)
    const double us =
        f.us_else + (double)steps * us_step + us_part * (double)parts;
    if (parts > 1 && us < least) {
      least = us;
      best.parts = (int)parts;
      best.steps = (int)steps;
      best.kernel = f.kernel;
    }
  }
}
// The time of a product over K, a multiple of 16, and how it is split.
double product_us(const Sizes &p, GemmSplit &best) {
  double least = 0.0;
  (void)choose_tile(p, &least);
  if (!split_possible(p, false))
    return least;
  try_split(kSplitBs, p, best, least);
  if (p.K % kGemmBK == 0) {
    try_split(kSplitDma128, p, best, least);
    if (p.N > 64)
      try_split(kSplitDma64, p, best, least);
  }
  return least;
}
// And in k_gemm_i8, for any K: tiles of 128 x 128 and of 64 x 128, three blocks of
// which run on a CU and are dealt out more evenly; the model of kTileCosts.  Its
// times are compared with those of other ways, so that they, kSplitAny's and the
// copy's (gemm_padded_k) are fitted together, to the times themselves and to the
// choice: to two thirds of 1294 products of awkward rows of up to 8.3e10
// multiply-adds, each timed in both tiles, with its rows copied and in up to ten
// splits (profiles/awkward_row_times.csv).  What is chosen takes 0.6 % longer than the
// fastest way in the geometric mean, on the third that was left out as on the rest, and
// 0.5 % above 26 us; the times are within 8 %, root mean square.  (Fitted to the choice
// between the two tiles alone, and to products of up to 26 us, long ones were thought
// 11 % too fast and left where they lie: 2.1 %, above 26 us 9 %.)
double any_us(bool low, const Sizes &p) {
  static constexpr TileCost t128 = {kT128x128, 128, 128, 1, 0.527, 0.350, 0.239,
      2.419, 2.531, 1.932, 0.390};
  static constexpr TileCost t64 = {kT128x128, 64, 128, 1, 0.219, 0.198, 0.214,
      1.126, 1.180, 2.398, 0.305};
  return tile_us(low ? t64 : t128, p);
}
bool any_takes_64_rows(const Sizes &p) {
  return any_us(true, p) < any_us(false, p);
}
double general_us(const Sizes &p, GemmSplit &best) {
  double least = std::min(any_us(false, p), any_us(true, p));
  if (split_possible(p, true))
    try_split(kSplitAny, p, best, least);
  return least;
}
GemmSplit split_plan(const GemmArgs &g, int a_mode) {
  GemmSplit best;
  const bool any = !gemm_fast_path(g.M, g.K, g.A);
  const Sizes p = sizes_of(g);
  if (g.X || g.M * g.N <= 0 || !split_possible(p, any) ||
      skinny_ok(g.M, g.K))
    return best;
  if (!any && g.K % 64 == 0 &&
      (flight_ok(g, a_mode) || (wreg_ok(g) && wreg_pays(g.M, g.N))))
    return best;
  const char *force = getenv("OM_MI355X_GEMM_TILE");
  if (force && force[0])
    return best;
  if (any)
    (void)general_us(p, best);
  else
    (void)product_us(p, best);
  return best;
}

const char *dma_name(bool narrow, bool ragged) {
  return narrow ? (ragged ? "k_gemm_i8_dma (128x64 tiles, ragged K)"
                          : "k_gemm_i8_dma (128x64 tiles)")
                : (ragged ? "k_gemm_i8_dma (128x128 tiles, ragged K)"
                          : "k_gemm_i8_dma (128x128 tiles)");
}

template <int A_MODE, int EPI>
hipError_t launch_split(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  const GemmSplit &p = g.split;
  const int M = (int)g.M, N = (int)g.N;
  EpiParams pe = ep;
  pe.out = g.parts;
  hipError_t e;
  if (p.kernel == kSplitBs) {
    e = launch_gemm_bs_split(st, g, pe, A_MODE);
  } else {
    const bool narrow = p.kernel == kSplitDma64;
    const int tiles_m = (M + 127) / 128;
    const int tiles_n = narrow ? (N + 63) / 64 : (N + 127) / 128;
    const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)p.parts);
    t_last_kernel = p.kernel == kSplitAny
                        ? "k_gemm_i8 (any K, any alignment; split along K)"
                    : narrow ? "k_gemm_i8_dma (128x64 tiles, split along K)"
                             : "k_gemm_i8_dma (128x128 tiles, split along K)";
    if (p.kernel == kSplitAny)
      k_gemm_i8<128, 128, 2, 2, 2, A_MODE, kEpiI32, kLoadAny, true>
          <<<grid, 256, 0, st>>>(tile_args(g, pe, kEpiI32));
    else if (narrow)
      k_gemm_i8_dma<64, 3, 3, A_MODE, kEpiI32, false, true><<<grid, 256, 0, st>>>(tile_args(g, pe, kEpiI32));
    else
      k_gemm_i8_dma<128, 3, 3, A_MODE, kEpiI32, false, true><<<grid, 256, 0, st>>>(tile_args(g, pe, kEpiI32));
    e = hipGetLastError();
  }
  if (e != hipSuccess)
    return e;
  const unsigned n = (unsigned)(g.M * g.N);
  const bool vec = (((uintptr_t)g.out) & (EPI == kEpiQ8 ? 3 : 15)) == 0;
  k_sum_parts<EPI><<<(n + 1023) / 1024, 256, 0, st>>>(
      SumArgs{g.parts, p.parts, n, (unsigned)N, vec, pack_epi(ep, EPI)});
  return hipGetLastError();
}

// k_gemm_i8_dma in tiles of 128 columns or, for cfg = kD128x64, of 64.
template <int A_MODE, int EPI>
hipError_t launch_dma(hipStream_t st, const GemmArgs &g, const EpiParams &ep,
    int cfg) {
  const int tiles_m = (int)((g.M + 127) / 128);
  const int N = (int)g.N, K = (int)g.K;
  const bool narrow = cfg == kD128x64, ragged = K % BK != 0;
  const int tiles_n = narrow ? (N + 63) / 64 : (N + 127) / 128;
  t_last_kernel = dma_name(narrow, ragged);
  auto *const kernel =
      narrow ? (ragged ? k_gemm_i8_dma<64, 3, 3, A_MODE, EPI, true>
                       : k_gemm_i8_dma<64, 3, 3, A_MODE, EPI, false>)
             : (ragged ? k_gemm_i8_dma<128, 3, 3, A_MODE, EPI, true>
                       : k_gemm_i8_dma<128, 3, 3, A_MODE, EPI, false>);
  kernel<<<dim3((unsigned)(tiles_m * tiles_n)), 256, 0, st>>>(tile_args(g, ep, EPI));
  return hipGetLastError();
}

template <int A_MODE, int EPI>
hipError_t gemm_launch_cfg(
    hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  const char *force = getenv("OM_MI355X_GEMM_TILE");
  if (g.X) {
    // rows quantized inside the kernel (the caller asked gemm_quantizes_rows)
    if (A_MODE != 2 || !gemm_quantizes_rows(g.M, g.K, g.N, g.X))
      return hipErrorInvalidValue;
    if (!skinny_quantizes_rows(g.M, g.K, g.X)) {
      // more rows than every block can quantize for itself: the blocks share
      // the minimum / maximum through the exchange slots
      if (EPI != kEpiF32 || !g.dql)
        return hipErrorInvalidValue;
      t_last_kernel = "k_gemm_i8_flight (rows quantized in the kernel)";
      t_limits_written = ep.limits.out != nullptr; // and reduces their limits
      return launch_gemm_flight_dq(st, g, ep, *g.dql);
    }
    return launch_gemm_skinny(st, g, ep, A_MODE);
  }
  // Up to 64 rows the weight-streaming kernel is ahead of every tile kernel
  // (K=4096 N=11008: M=33 11.6 against 17.2 us, M=48 12.3 / 17.7; K=11008
  // N=4096 M=64: 15.0 / 37.7; K=768 N=3072 M=64: 4.2 / 6.0).
  if (skinny_ok(g.M, g.K) && !(force && force[0]))
    return launch_gemm_skinny(st, g, ep, A_MODE);
  if (g.parts && g.split.parts > 1)
    return launch_split<A_MODE, EPI>(st, g, ep);
  const int tiles_m = (int)((g.M + 127) / 128);
  const int tiles_n128 = (int)((g.N + 127) / 128);
  if (!gemm_fast_path(g.M, g.K, g.A)) {
    // Any K, any alignment of A (and the forced configurations of the tests
    // when M <= 16); byte loads only for an A of fewer than 16 bytes.
    const bool low = g.M * g.K >= 16 && any_takes_64_rows(sizes_of(g));
    t_last_kernel = low ? "k_gemm_i8 (any K, any alignment; 64x128 tiles)"
                        : "k_gemm_i8 (any K, any alignment)";
    const int tiles_m64 = (int)((g.M + 63) / 64);
    if (low)
      k_gemm_i8<64, 128, 2, 2, 3, A_MODE, EPI, kLoadAny>
          <<<dim3((unsigned)(tiles_m64 * tiles_n128)), 256, 0, st>>>(tile_args(g, ep, EPI));
    else if (g.M * g.K >= 16)
      k_gemm_i8<128, 128, 2, 2, 2, A_MODE, EPI, kLoadAny>
          <<<dim3((unsigned)(tiles_m * tiles_n128)), 256, 0, st>>>(tile_args(g, ep, EPI));
    else
      k_gemm_i8<128, 128, 2, 2, 2, A_MODE, EPI, kLoadBytes>
          <<<dim3((unsigned)(tiles_m * tiles_n128)), 256, 0, st>>>(tile_args(g, ep, EPI));
    return hipGetLastError();
  }
  const int cfg = choose_tile(sizes_of(g));
  if (g.K % 64 != 0 && cfg != kB64x256 && cfg != kB64x128)
    return launch_dma<A_MODE, EPI>(st, g, ep,
        cfg == kD128x64 || cfg == kD128x128 ? cfg : (int)kD128x128);
  // One round of blocks with everything requested at once: small problems,
  // where a pipelined K loop would pay the memory latency step after step
  // (512 x 1024 x 4096 QLinearMatMul: 8.2 us in 128 x 64 tiles of
  // k_gemm_i8_dma; 128 x 768 x 768: 7.0 us).
  if ((cfg == kFlight || !(force && force[0])) && flight_ok(g, A_MODE)) {
    t_last_kernel = "k_gemm_i8_flight (one round, operands requested at once)";
    t_limits_written = EPI == kEpiF32 && ep.limits.out != nullptr;
    return launch_gemm_flight(st, g, ep, A_MODE);
  }
  // Weights in registers: K = 768 (the projections of a BERT-base layer)
  // when the problem fills the device with its 128 x 384 blocks.
  const bool forced = force && force[0];
  if (wreg_ok(g) && (cfg == kW128x384 || (!forced && wreg_pays(g.M, g.N)))) {
    t_last_kernel = "k_gemm_i8_wreg (weights in registers, 128x384 blocks)";
    // (the limits of y: in the kernel for the f32 results of a fused layer)
    t_limits_written = A_MODE == 2 && EPI == kEpiF32 && ep.limits.out != nullptr;
    return launch_gemm_wreg(st, g, ep, A_MODE);
  }
  switch (cfg) {
  case kB128x256:
  case kB64x256:
  case kB64x128: {
    const BsTile tile = cfg == kB128x256  ? kBs128x256
                        : cfg == kB64x256 ? kBs64x256
                                          : kBs64x128;
    if (!bs_ok(g, tile)) // (forced, on a K this kernel does not take)
      return launch_dma<A_MODE, EPI>(st, g, ep, kD128x128);
    return launch_gemm_bs(st, g, ep, A_MODE, tile);
  }
  case kD128x64:
    return launch_dma<A_MODE, EPI>(st, g, ep, kD128x64);
  case kW128x384: // (forced, on a shape that kernel does not take)
  case kFlight:
  case kD128x128:
    return launch_dma<A_MODE, EPI>(st, g, ep, kD128x128);
  default:
    t_last_kernel = "k_gemm_i8 (128x128 tiles through registers)";
    k_gemm_i8<128, 128, 2, 2, 2, A_MODE, EPI, kLoadAligned>
        <<<dim3((unsigned)(tiles_m * tiles_n128)), 256, 0, st>>>(tile_args(g, ep, EPI));
    break;
  }
  return hipGetLastError();
}

template <int A_MODE>
hipError_t gemm_launch_epi(
    hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  switch (g.epi) {
  case kEpiI32:
    return gemm_launch_cfg<A_MODE, kEpiI32>(st, g, ep);
  case kEpiF32:
    return gemm_launch_cfg<A_MODE, kEpiF32>(st, g, ep);
  default:
    return gemm_launch_cfg<A_MODE, kEpiQ8>(st, g, ep);
  }
}

// Rows of A copied to a pitch of Kp >= K bytes, a multiple of 16, the bytes past
// K set to the row's zero point (exclusive-ored with `flip`: 0x80 for rows stored
// minus 128): an element equal to its zero point stands for the real value 0, so
// a product over the Kp bytes equals the product over the K (see gemm_padded_k).
// 16 bytes of the result per thread, read at whatever address they have (M * K
// >= 16; moved back to end with A where they would run past it).  Bound by the
// launch and by memory: 4096 x 1000 in 3.4 us.
__global__ __launch_bounds__(256) void k_pad_rows(const uint8_t *__restrict__ A,
    unsigned M, unsigned K, unsigned chunks, const uint8_t *__restrict__ zp,
    int zp_len, uint8_t flip, uint8_t *__restrict__ out) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= M * chunks)
    return;
  const unsigned r = i / chunks, c = i - r * chunks;
  const bool has_zp = zp && zp_len > 0;
  const uint8_t z = (has_zp ? zp : A)[has_zp && zp_len > 1 ? r : 0];
  const uint8_t *const p = A + (uint64_t)r * K + c * 16;
  const uint8_t *const last = A + ((uint64_t)M * K - 16);
  const v4i v = *(const v4i_any *)(p < last ? p : last);
  const int left = (int)K - (int)(c * 16);
  const int len = left < 0 ? 0 : left < 16 ? left : 16;
  const uint64_t fill =
      (uint64_t)(uint8_t)((has_zp ? z : 0) ^ flip) * 0x0101010101010101ull;
  *(v4i *)(out + (uint64_t)i * 16) =
      row_chunk(v, p < last ? 0 : (int)(p - last), len, fill);
}

} // namespace

// Rows (more than 64) whose length is no multiple of 16 bytes, or that do not start
// on a 16-byte boundary, leave k_gemm_i8, at half the speed of the other kernels.
// The runtime copies such rows to an aligned buffer first, with as many bytes as
// this says (0: not), the tail of each row filled with its zero point, and
// multiplies with that K: (a - a_zp) is zero there, so the products, the row sums
// and the K * (a offset) * (b offset) term of the zero-point algebra are those of
// the original rows, bit for bit.  Where the copy -- 2.9 us and two ways through
// memory, by the fit of any_us -- costs less than it saves: int32 1178 x 4084 x 8832
// 74.5 us as it lies, 58.5 copied, f32 with row sums 4095 x 2749 x 2584 59.1 / 49.2, u8
// 1905 x 7689 x 1664 49.4 / 41.7; left alone: int32 with row sums 4099 x 777 x 1001 13.6 /
// 17.3, u8 575 x 948 x 8448 13.7 / 15.2.
int64_t gemm_padded_k(const GemmArgs &g) {
  const char *force = getenv("OM_MI355X_GEMM_TILE");
  const int64_t M = g.M, K = g.K, N = g.N;
  if (M < 1 || K < 1 || N < 1 ||
      (K % 16 == 0 && (((uintptr_t)g.A) & 15) == 0) || (force && force[0]))
    return 0;
  // k_gemm_i8_skinny takes such rows as they are.  Where it reads many bytes at
  // addresses that are no multiple of 4, or any in more than one round of blocks,
  // that costs more than the copy's 3 us (893 products timed both ways,
  // profiles/few_row_times.csv: 0.2 % above always taking the faster; 2.1 % never
  // copying, 2 % copying 33 rows and more from K = 4096 on).  As they lie / copied:
  //  - more than 32 rows and 256 blocks of 32 columns: 50 x 1137 x 9152 13.3 / 9.2
  //    us, 53 x 312 x 10560 9.2 / 7.2;
  //  - 120 KB in rows that start between such addresses, with up to 32 rows only if
  //    all do: 43 x 9313 x 1792 (three rows of four) 16.4 / 12.8, 54 x 4604 x 3232 (two
  //    bytes off) 13.3 / 9.7, but 19 x 2938 x 4032 5.3 / 6.9, 62 x 8552 x 328 (none) 10.4 /
  //    15.5, 32 x 8022 x 5616 (one of two) 10.7 / 13.0.
  if (M <= 64) {
    int64_t odd = 0; // of four rows in turn
    for (uintptr_t r = 0; r < 4; ++r)
      odd += (((uintptr_t)g.A + r * (uintptr_t)K) & 3) != 0;
    const bool many = odd * M * K > 480000 && (M > 32 || odd == 4);
    return many || (M > 32 && N > 8192) ? round_up(K, 16) : 0;
  }
  const int64_t Kp = round_up(K, kGemmBK);
  if (Kp >= (1 << 24) || M * (Kp / 16) > UINT32_MAX || M > INT32_MAX ||
      N > INT32_MAX)
    return 0;
  GemmSplit s1, s2;
  const Sizes own = sizes_of(g);
  Sizes padded = own;
  padded.K = Kp;
  double us = product_us(padded, s1);
  // (k_gemm_i8_flight, one round of 64 x 128 blocks)
  if ((Kp == 512 || Kp == 768 || Kp == 1024) &&
      ((M + 63) / 64) * ((N + 127) / 128) <= 256)
    us = std::min(us, 2.4 + 0.002 * (double)Kp);
  return general_us(own, s2) > us + 2.9 + 3.6e-7 * (double)(M * K) ? Kp : 0;
}

hipError_t launch_pad_rows(hipStream_t s, const void *a, int64_t M, int64_t K,
    int64_t Kp, const void *a_zp, int64_t a_zp_len, bool stored_minus_128,
    void *out) {
  const int64_t n = M * (Kp / 16);
  if (M * K < 16 || Kp < K || Kp % 16 != 0 || Kp > INT32_MAX || n > UINT32_MAX)
    return hipErrorInvalidValue;
  k_pad_rows<<<(unsigned)((n + 255) / 256), 256, 0, s>>>((const uint8_t *)a,
      (unsigned)M, (unsigned)K, (unsigned)(Kp / 16), (const uint8_t *)a_zp,
      (int)a_zp_len, stored_minus_128 ? 0x80 : 0, (uint8_t *)out);
  return hipGetLastError();
}

hipError_t launch_pack_b(hipStream_t s, const void *B, bool b_unsigned,
    int64_t K, int64_t N, int8_t *Bp, int32_t *colsum) {
  const int64_t Kpad = round_up(K > 0 ? K : 1, kGemmBK);
  const int64_t Npad = round_up(N, kGemmBN);
  hipError_t e = launch_fill_u32(s, (uint32_t *)colsum, Npad, 0u);
  if (e != hipSuccess)
    return e;
  // kGemmBK and kGemmBN are multiples of the 64 x 64 pack tile, so the grid
  // covers [Npad, Kpad] exactly and every byte of Bp is written.
  const int KT = (int)(Kpad / kGemmBK);
  dim3 grid((unsigned)(Npad / PT), (unsigned)(Kpad / PT));
  if (b_unsigned)
    k_pack_b<true><<<grid, 256, 0, s>>>(
        (const uint8_t *)B, K, N, KT, Bp, colsum);
  else
    k_pack_b<false><<<grid, 256, 0, s>>>(
        (const uint8_t *)B, K, N, KT, Bp, colsum);
  return hipGetLastError();
}

int gemm_quantizes_rows(int64_t M, int64_t K, int64_t N, const void *x) {
  const char *force = getenv("OM_MI355X_GEMM_TILE");
  if (force && force[0])
    return 0;
  if (skinny_quantizes_rows(M, K, x))
    return 1;
  return flight_quantizes_rows(M, K, N, x) ? 2 : 0;
}

size_t gemm_plan_split(GemmArgs &g) {
  g.split = split_plan(g, (g.X || g.a_preshifted) ? 2 : (g.a_unsigned ? 1 : 0));
  return g.split.parts > 1 ? (size_t)g.split.parts * part_stride(g) * 4 : 0;
}

const char *last_gemm_kernel() { return t_last_kernel; }
void note_gemm_kernel(const char *name) { t_last_kernel = name; }

hipError_t launch_gemm(hipStream_t s, const GemmArgs &g) {
  if (g.M == 0 || g.N == 0)
    return hipSuccess;
  if (g.M > INT32_MAX || g.N > INT32_MAX || g.K > INT32_MAX ||
      g.M * g.N > ((int64_t)1 << 40))
    return hipErrorInvalidValue;
  EpiParams ep;
  ep.a_zp = g.a_zp;
  ep.a_zp_len = g.a_zp ? g.a_zp_len : 0;
  ep.b_zp = g.b_zp;
  ep.b_zp_len = g.b_zp ? g.b_zp_len : 0;
  ep.need_rowsum = g.b_unsigned || (g.b_zp != nullptr && g.b_zp_len > 0);
  ep.colsum = g.colsum;
  ep.a_scale = g.a_scale;
  ep.b_scale = g.b_scale;
  ep.b_scale_len = g.b_scale_len;
  ep.y_scale = g.y_scale;
  ep.y_zp = g.y_zp;
  ep.bias = g.epi == kEpiF32 ? g.bias : nullptr;
  ep.bias_len = g.bias_len;
  ep.x_limits = g.X ? g.x_limits : nullptr;
  ep.limits = LimitsOut{};
  if (g.y_limits) // (slot [4] of the counters: [0] is DynamicQuantizeLinear's)
    ep.limits = LimitsOut{g.y_limits, g.dql->partial_min, g.dql->partial_max,
        g.dql->counter + 4};
  ep.floor = relu_floor(g.epi == kEpiF32 && g.relu);
  ep.gelu = g.epi == kEpiF32 && g.gelu;
  ep.out = g.out;
  ep.b_unsigned = g.b_unsigned;
  ep.y_unsigned = g.y_unsigned;
  ep.narrow = (int)g.narrow;
  const int a_mode = (g.X || g.a_preshifted) ? 2 : (g.a_unsigned ? 1 : 0);
  t_limits_written = false;
  if (g.y_limits && (g.epi != kEpiF32 || !g.dql))
    return hipErrorInvalidValue;
  hipError_t e;
  switch (a_mode) {
  case 0:
    e = gemm_launch_epi<0>(s, g, ep);
    break;
  case 1:
    e = gemm_launch_epi<1>(s, g, ep);
    break;
  default:
    e = gemm_launch_epi<2>(s, g, ep);
    break;
  }
  if (e == hipSuccess && g.y_limits && !t_limits_written)
    e = launch_minmax_limits(s, *g.dql, (const float *)g.out, g.M * g.N, g.y_limits);
  return e;
}


} // namespace om
