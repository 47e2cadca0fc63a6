// int8 GEMM with the weights streamed from Bp straight into MFMA operand
// registers.  What is computed, and the layout of Bp, are described at the top
// of gemm_kernels.hip.
//
// Bp is stored in exactly the order the matrix cores consume it: the operand of
// column tile nt, K step ks, half step sub is one contiguous KiB, 16 bytes per
// lane.  The four waves of a block sit side by side along N; each owns 32*TN
// columns that no other wave needs and loads their operands into registers,
// three steps ahead.  Only the A tile, which all four waves share, goes through
// LDS, copied there without passing through registers.
//
// What bounds it: the lines a CU can have on their way, about 64 of 128 bytes,
// each some 300 clocks away (2048 x 11008 x 4096: 8.56 million line requests of
// 297 clocks, 58 of them in flight per CU throughout, the matrix cores busy half
// of the time).  So:
//  - A is copied in stages of two K steps, a row's piece being one whole line
//    (pieces of 64 bytes fetched most lines twice: 10.0 million requests);
//  - what lies past the last step is asked for with empty descriptors, which
//    move nothing and count like any other load;
//  - a block asks for little in front of its loop (below).
// Registers let two blocks of 128 x 256 run on a CU, three of 64 x 256 and four
// of 64 x 128.
#include "gemm_common.h"
#include "gemm_epilogue.h"

namespace om {
namespace gemm {

namespace {

// SPLIT: the block multiplies blockIdx.y's part of K only (KSplit).
// RAGGED: K is a multiple of 16 but not of a K step: the row sums leave out what
// lies past the end of the row (the weights are zero there).
template <int TM, int TN, int A_MODE, int EPI, bool RS, bool RAGGED, bool SPLIT>
__device__ __forceinline__ void stream_tile(const uint8_t *__restrict__ A,
    const int8_t *__restrict__ Bp, int M, int N, int K, int Kpad,
    const EpiParams &ep, int tiles_m, int tiles_n, const KSplit &ks) {
  constexpr int D = 4;   // sets of weights registers
  constexpr int NST = 4; // stages of A in LDS
  constexpr int BM = 32 * TM, BN = 4 * 32 * TN;
  constexpr int ROW = 2 * BK;         // bytes of a row in a stage: two K steps
  constexpr int STAGE = BM * ROW;
  constexpr int CA = BM / 32; // A copies (1 KiB each) per wave and stage
  static_assert(BM % 64 == 0, "tile height");
  __shared__ __attribute__((aligned(1024))) uint8_t sm[NST * STAGE];

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
  const int l32 = lane & 31;
  const int lh = lane >> 5;
  const int ncol0 = n0 + wave * 32 * TN;

  const int KTs = Kpad / BK; // K steps of the operands, and of this block
  const int kfirst = SPLIT ? (int)blockIdx.y * ks.steps : 0;
  const int KT = SPLIT && ks.steps < KTs - kfirst ? ks.steps : KTs - kfirst;

  // A copies: copy j of a stage fills LDS bytes [j*1024, (j+1)*1024) of it,
  // lane -> row j*8 + lane/8, holding chunk (lane%8) ^ ((row/2)%8) of the row's
  // 128 bytes: sixteen consecutive rows (two to each turn of the 64 banks) then
  // hold any one chunk in sixteen different places, which is what an operand
  // read needs.  By descriptor (tile origin), a 32-bit lane offset that does not
  // change from stage to stage and the stage as scalar offset: no vector address
  // arithmetic in the loop.
  const int crow = lane >> 3;
  uint32_t ga[CA];
#pragma unroll
  for (int h = 0; h < CA; ++h) {
    const int r = (wave * CA + h) * 8 + crow;
    const int rc = (m0 + r < M) ? r : M - 1 - m0; // rows past M: never stored
    ga[h] = (uint32_t)rc * (uint32_t)K +
            (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u;
  }
  typedef __attribute__((address_space(3))) void *lds_ptr;
  const int a_bytes = (M - m0 < BM ? M - m0 : BM) * K - kfirst * BK;
  const uint8_t *const a_tile =
      scalar_ptr(A + (int64_t)m0 * K + (int64_t)kfirst * BK);
  auto copy_a = [&](int pair, int stage) {
    uint8_t *base = sm + stage * STAGE + wave * CA * 1024;
    const bool in = pair * 2 < KT;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)a_tile, 0, in ? a_bytes : 0, 0x00020000);
    const int soff = in ? pair * ROW : 0;
#pragma unroll
    for (int h = 0; h < CA; ++h)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (lds_ptr)(base + h * 1024), 16, (int)ga[h], soff, 0, 0);
  };

  // Bp operands of this wave's column tiles, by buffer addressing: one
  // descriptor in scalar registers, a 32-bit lane offset, and the step as a
  // scalar offset.  The loads are written as inline assembly because the
  // compiler, which cannot count memory operations across the loop's back
  // edge, would otherwise wait for every outstanding one (vmcnt(0)) before
  // the first use of these registers in each trip, draining the prefetch.
  v4i brsrc;
  {
    const uint64_t a =
        (uint64_t)(Bp + ((int64_t)(ncol0 >> 5) * KTs + kfirst) * 2048);
    brsrc.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    brsrc.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu));
    brsrc.z = 0;          // bytes covered: set per step
    brsrc.w = 0x00020000; // raw buffer, 32-bit elements
  }
  const int b_bytes = (TN - 1) * KTs * 2048 + KT * 2048;
  int boff[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    boff[j] = j * KTs * 2048 + lane * 16;
  int bstep = 0;
  auto weights_of = [&](int step) { // the step that load_b asks for
    brsrc.z = step < KT ? b_bytes : 0;
    bstep = step < KT ? step * 2048 : 0;
  };
  // (The half step is in the instruction: the device compares the other offsets
  // with the descriptor's size minus the scalar one, unsigned, so that an empty
  // descriptor asks for nothing only with a scalar offset of 0.)
  using Half0 = std::integral_constant<int, 0>;
  using Half1 = std::integral_constant<int, 1>;
  auto load_b = [&](auto half, v4i(&fb)[TN]) {
    // (named here: asm operands alone do not capture in a generic lambda)
    const int soff = bstep;
    const v4i rsrc = brsrc;
    const int(&off)[TN] = boff;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:%4"
                   : "=v"(fb[j])
                   : "v"(off[j]), "s"(rsrc), "s"(soff),
                   "n"(decltype(half)::value * 1024)
                   : "memory");
  };

  // A operand reads: half step h (0 .. 3) of a stage uses chunk 2*h + lane/32
  // of row lane%32 of MFMA row tile i (32 * ROW bytes apart).
  const unsigned sm_base = (unsigned)(uintptr_t)(lds_ptr)sm;
  // (sm_base is a multiple of 128: bits 4 .. 6 are the chunk's)
  const unsigned ra = sm_base + l32 * ROW + ((lh ^ ((l32 >> 1) & 7)) << 4);
  auto lds_read = [](v4i &f, unsigned addr, auto off) {
    asm volatile("ds_read_b128 %0, %1 offset:%2"
                 : "=v"(f)
                 : "v"(addr), "n"(decltype(off)::value)
                 : "memory");
  };
  auto read_a = [&](v4i(&f)[TM], int h, unsigned soff) {
    const unsigned at = (ra ^ (unsigned)(h << 5)) + soff;
    static_for<TM>([&](auto i) {
      lds_read(f[decltype(i)::value], at,
          std::integral_constant<int, decltype(i)::value * 32 * ROW>{});
    });
  };

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0;

  // Vector memory operations of a wave, in issue order, for every pair of
  // steps p (CB = 2 * TN weights loads a step):
  //   step 2p:     CA copies of pair p+2, CB weights of step 2p+3
  //   step 2p+1:   CB weights of step 2p+4
  // and, before the loop, what pairs -2 and -1 would have asked for.  They
  // complete in order, so a wait for "all but the youngest n" is exact:
  //   top of step 2p: its weights were asked for in step 2p-3; younger: those
  //     of 2p+1 and 2p+2 and the copies of pair p+1 (2 * CB + CA)
  //   top of step 2p+1: its weights were asked for in step 2p-2, behind the
  //     copies of pair p+1, which are read from the second half of this step
  //     on; younger: the weights of 2p+2 and 2p+3 and the copies of pair p+2
  // No more than this on its way: a wave cannot start before it has issued
  // everything in front of the loop, and the path into the CU takes a load in 64
  // clocks (weights four steps ahead and copies half a pair earlier, 128 x 256
  // tiles: 2048 x 768 x 4096 12.9 us, 11.6 so).
  // The barrier is at the top of step 2p+1 only: behind it every wave's copies
  // of pair p+1 are in LDS, and every wave is done with pair p-1 (its last
  // operands were waited for in step 2p-1), whose stage the copies issued in
  // step 2p+2, of pair p+3, overwrite.
  constexpr int CB = 2 * TN;
  constexpr int kYoung = 2 * CB + CA;
  static_assert(3 * CB + 2 * CA < 64, "wait count");
  v4i bs[D][2][TN];
  copy_a(0, 0);
#pragma unroll
  for (int u = 0; u < D - 1; ++u) {
    weights_of(u);
    load_b(Half0{}, bs[u][0]);
    load_b(Half1{}, bs[u][1]);
    if (u == 0)
      copy_a(1, 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  const v4i flip = {(int)0x80808080, (int)0x80808080, (int)0x80808080,
      (int)0x80808080};

  // RS: row sums of A are needed (B carries an offset).  The four waves have the
  // same rows: each sums one of the four half steps of a pair, and they add up
  // through LDS behind the loop.  (All of them in every wave: uint8 B, 64 x 128
  // tiles, 85 x 6336 x 10560 28.4 us, 128 x 6464 x 9637 29.6; so 23.1, 24.1; without
  // row sums 20.2, 21.3.)
  constexpr int RC = TM == 2 ? 4 : 1; // (independent sums, where registers are left)
  int32_t rsp[TM][RC];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int c = 0; c < RC; ++c)
      rsp[i][c] = 0;
  // Bytes of a row from this lane's chunk of this block's first step on.
  const int row_left =
      (K < (kfirst + KT) * BK ? K : (kfirst + KT) * BK) - kfirst * BK - lh * 16;
  auto wait_vm = [](auto n) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (decltype(n)::value & 15) |
                               ((decltype(n)::value >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto wait_first = [] { // the operands read before the last TM ones
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(%0)" : : "n"(TM) : "memory");
  };
  auto mfmas = [&](v4i(&fa)[TM], v4i(&fb)[TN], int step, int step_in_pair,
                   int half) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      asm volatile("" : "+v"(fa[i])); // written here, behind the wait
    if (A_MODE == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[i] ^= flip;
    }
    if (RS && wave == (step_in_pair * 2 + half)) {
      // (a step past the last one: its operands are whatever LDS holds)
      const int ones =
          (RAGGED ? step * BK + half * 32 < row_left : step < KT) ? 0x01010101 : 0;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          rsp[i][c % RC] = __builtin_amdgcn_sdot4(fa[i][c], ones, rsp[i][c % RC], false);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
            fa[i], fb[j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };

  // The copies of pair 0 (the oldest) have landed, of every wave.
  wait_vm(std::integral_constant<int, 3 * CB + CA>{});
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  v4i fa0[TM];
  read_a(fa0, 0, 0);
  int stage = 0;
  // Two K steps.  Operands are read one half step early: those of the second
  // half while the first half's MFMAs run, and those of the next step's first
  // half while the second half's do, so that no MFMA waits for an LDS read
  // issued just before it.  Loads are issued in front of the MFMAs (behind them
  // they waited for the matrix cores: 1024 x 4096 x 4096 29.4 / 28.3 us).
  auto pair = [&](int kt, auto u_c) {
    constexpr int u = decltype(u_c)::value;
    constexpr int v = (u + D - 1) % D; // set of the weights asked for in step u
    const unsigned soff = (unsigned)(stage * STAGE);
    const int nstage = (stage + 1) & (NST - 1);
    v4i fa1[TM], fb0[TM], fb1[TM];
    wait_vm(std::integral_constant<int, kYoung>{});
    read_a(fa1, 1, soff);
    copy_a((kt >> 1) + NST - 2, (stage + NST - 2) & (NST - 1));
    weights_of(kt + D - 1);
    load_b(Half0{}, bs[v][0]);
    wait_first();
    mfmas(fa0, bs[u][0], kt, 0, 0);
    read_a(fb0, 2, soff);
    load_b(Half1{}, bs[v][1]);
    wait_first();
    mfmas(fa1, bs[u][1], kt, 0, 1);

    wait_vm(std::integral_constant<int, kYoung>{});
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read_a(fb1, 3, soff);
    weights_of(kt + D);
    load_b(Half0{}, bs[u][0]);
    wait_first();
    mfmas(fb0, bs[u + 1][0], kt + 1, 1, 0);
    read_a(fa0, 0, (unsigned)(nstage * STAGE));
    load_b(Half1{}, bs[u][1]);
    wait_first();
    mfmas(fb1, bs[u + 1][1], kt + 1, 1, 1);
    stage = nstage;
  };
  // Whole trips of four steps, one way out: steps past the last one multiply
  // zeros.  (Leaving after the first pair as well made the compiler move the
  // accumulators through scratch memory.)
  for (int kt = 0; kt < KT; kt += D) {
    pair(kt, std::integral_constant<int, 0>{});
    pair(kt + 2, std::integral_constant<int, 2>{});
  }
  // What was asked for past the last step has still to come back, and its
  // registers count as used here: nothing else is put there before.
  __builtin_amdgcn_s_waitcnt(0x0070); // vmcnt(0) lgkmcnt(0)
#pragma unroll
  for (int u = 0; u < D; ++u)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      asm volatile("" : : "v"(bs[u][0][j]), "v"(bs[u][1][j]) : "memory");
#pragma unroll
  for (int i = 0; i < TM; ++i)
    asm volatile("" : : "v"(fa0[i]) : "memory");
  __builtin_amdgcn_sched_barrier(0);

  int32_t rsum[TM] = {};
  if (RS) {
    // (nobody reads operands any more behind the first barrier)
    int32_t(*const sums)[TM][64] = (int32_t(*)[TM][64])sm;
    lds_barrier();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      int32_t own = rsp[i][0];
#pragma unroll
      for (int c = 1; c < RC; ++c)
        own += rsp[i][c];
      sums[wave][i][lane] = own;
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < TM; ++i)
      rsum[i] = sums[0][i][lane] + sums[1][i][lane] + sums[2][i][lane] +
                sums[3][i][lane];
  }

  EpiParams e = ep;
  if (SPLIT)
    e = part_of(ep, ks);
  e.need_rowsum = RS; // known here: the other form's code goes
  constexpr int kAux = SPLIT ? 0 : kAuxThrough;
  const bool whole_k = !SPLIT || blockIdx.y == 0;
  gemm_epilogue<TM, TN, A_MODE, EPI, kAux>(
      acc, rsum, m0, ncol0, M, N, whole_k ? K : 0, e, whole_k);
}

// 128 x 256 tiles.
template <int A_MODE, int EPI, bool RS>
__global__ __launch_bounds__(256, 2) void k_gemm_i8_bs(TileArgs a) {
  stream_tile<4, 2, A_MODE, EPI, RS, false, false>(a.A, a.Bp, a.M, a.N, a.K,
      padded_k(a.K), unpack_epi<EPI>(a.epi), tiles_of(a.M, 128), tiles_of(a.N, 256),
      KSplit{});
}
// 64 x 256 and 64 x 128 tiles.
template <int TN, int MINB, int A_MODE, int EPI, bool RS, bool RAGGED, bool SPLIT>
__global__ __launch_bounds__(256, MINB) void k_gemm_i8_dma_bs(TileArgs a) {
  stream_tile<2, TN, A_MODE, EPI, RS, RAGGED, SPLIT>(a.A, a.Bp, a.M, a.N, a.K,
      padded_k(a.K), unpack_epi<EPI>(a.epi), tiles_of(a.M, 64),
      tiles_of(a.N, 128 * TN), KSplit{a.steps, part_stride(a.M, a.N)});
}

// ragged: the form that looks for the end of the row (only row sums have to); in
// 64 x 256 tiles nothing is split.
const char *dma_bs_name(int tn, bool ragged, bool split) {
  if (tn == 2)
    return ragged ? "k_gemm_i8_dma_bs (64x256 tiles, ragged K)"
                  : "k_gemm_i8_dma_bs (64x256 tiles)";
  static const char *const names[2][2] = {
      {"k_gemm_i8_dma_bs (64x128 tiles)",
          "k_gemm_i8_dma_bs (64x128 tiles, split along K)"},
      {"k_gemm_i8_dma_bs (64x128 tiles, ragged K)",
          "k_gemm_i8_dma_bs (64x128 tiles, ragged K, split along K)"}};
  return names[ragged][split];
}

template <int TN, int A_MODE, int EPI, bool SPLIT>
void launch_dma_bs(hipStream_t st, const GemmArgs &g, const EpiParams &ep) {
  const int M = (int)g.M, N = (int)g.N, K = (int)g.K;
  const int tiles_m = (M + 63) / 64, tiles_n = (N + 128 * TN - 1) / (128 * TN);
  const bool ragged = ep.need_rowsum && K % BK != 0;
  constexpr int MINB = TN == 1 ? 4 : 3;
  note_gemm_kernel(dma_bs_name(TN, ragged, SPLIT));
  auto *const kernel =
      ep.need_rowsum
          ? (ragged ? k_gemm_i8_dma_bs<TN, MINB, A_MODE, EPI, true, true, SPLIT>
                    : k_gemm_i8_dma_bs<TN, MINB, A_MODE, EPI, true, false, SPLIT>)
          : k_gemm_i8_dma_bs<TN, MINB, A_MODE, EPI, false, false, SPLIT>;
  kernel<<<dim3((unsigned)(tiles_m * tiles_n), SPLIT ? (unsigned)g.split.parts : 1u),
      256, 0, st>>>(tile_args(g, ep, EPI));
}

template <int A_MODE, int EPI>
void launch_tile(hipStream_t st, const GemmArgs &g, const EpiParams &ep, BsTile tile) {
  if (tile == kBs64x128)
    return launch_dma_bs<1, A_MODE, EPI, false>(st, g, ep);
  if (tile == kBs64x256)
    return launch_dma_bs<2, A_MODE, EPI, false>(st, g, ep);
  const int M = (int)g.M, N = (int)g.N;
  const int tiles_m = (M + 127) / 128, tiles_n = (N + 255) / 256;
  note_gemm_kernel("k_gemm_i8_bs (128x256 tiles)");
  auto *const kernel = ep.need_rowsum ? k_gemm_i8_bs<A_MODE, EPI, true>
                                      : k_gemm_i8_bs<A_MODE, EPI, false>;
  kernel<<<dim3((unsigned)(tiles_m * tiles_n)), 256, 0, st>>>(tile_args(g, ep, EPI));
}

template <int A_MODE>
void launch_epi(hipStream_t st, const GemmArgs &g, const EpiParams &ep, BsTile tile) {
  if (g.epi == kEpiI32)
    launch_tile<A_MODE, kEpiI32>(st, g, ep, tile);
  else if (g.epi == kEpiF32)
    launch_tile<A_MODE, kEpiF32>(st, g, ep, tile);
  else
    launch_tile<A_MODE, kEpiQ8>(st, g, ep, tile);
}

} // namespace

// (K: the offsets of 128 rows and of two column tiles stay in 31 bits.)
bool bs_ok(const GemmArgs &g, BsTile tile) {
  return g.K > 0 && g.K < (1 << 24) && (((uintptr_t)g.A) & 15) == 0 &&
         g.K % (tile == kBs128x256 ? 4 * kGemmBK : 16) == 0;
}

hipError_t launch_gemm_bs(hipStream_t st, const GemmArgs &g, const EpiParams &ep,
    int a_mode, BsTile tile) {
  if (!bs_ok(g, tile))
    return hipErrorInvalidValue;
  if (a_mode == 0)
    launch_epi<0>(st, g, ep, tile);
  else if (a_mode == 1)
    launch_epi<1>(st, g, ep, tile);
  else
    launch_epi<2>(st, g, ep, tile);
  return hipGetLastError();
}

hipError_t launch_gemm_bs_split(hipStream_t st, const GemmArgs &g,
    const EpiParams &ep, int a_mode) {
  if (!bs_ok(g, kBs64x128))
    return hipErrorInvalidValue;
  if (a_mode == 0)
    launch_dma_bs<1, 0, kEpiI32, true>(st, g, ep);
  else if (a_mode == 1)
    launch_dma_bs<1, 1, kEpiI32, true>(st, g, ep);
  else
    launch_dma_bs<1, 2, kEpiI32, true>(st, g, ep);
  return hipGetLastError();
}

} // namespace gemm
} // namespace om
