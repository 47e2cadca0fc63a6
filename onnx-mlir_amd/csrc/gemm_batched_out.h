// How results leave k_gemm_i8_batched (gemm_batched.hip): the choice and the pieces
// that a tile is written in, as functions of sizes and addresses alone, which run on
// host and device.
#pragma once

#include <cstdint>

namespace om {
namespace gemm {

enum OutForm : int { kOutDirect, kOutTile, kOutRows };

// int32 results go by way of LDS where rows are no whole lines, in tiles as wide as the
// matrix and in rows of whole 16-byte pieces (not in other rows, whose ends are stores
// of their own: 64 x 511x64x511 17.2 us, 18.5 by LDS).  707 products timed both ways
// (profiles/batched_way_out_times.csv; us, direct / by LDS):
//   more than one block a CU: what a block writes then stands beside another's loads
//   (472x128x472 in 256 blocks 4.98 / 5.00, 320 5.72 / 5.50, 512 6.76 / 6.07; 64x64x100 in 256
//   4.28 / 4.36, 320 4.84 / 4.69, 768 7.67 / 6.05);
//   6 KB of results to a tile, for the barrier and the second way: below 2 KB 5 % slower
//   in the geometric mean, 2 to 6 KB 1.5 %, 6 to 8 KB 2 % faster, 8 to 20 KB 3 %, more 6 %;
//   up to 48 MB in all: up to 32 MB, the size of the L2s, 5 % faster, 32 to 48 MB 3 %; 48 to
//   75 MB 4 % slower (148 x 173x32x572 14.1 / 15.1).  Above that it depends on what the last-
//   level cache holds of the results that a program goes through: with three in turn 6 %
//   faster (0.68 to 1.10) to 110 MB, 18 % slower (0.70 to 1.54) beyond.
// 8-bit results do not: 2 % slower in the geometric mean of 173 products, up to 19 %.
// Results that do not start on a multiple of 4 are stored one by one: pieces of 16 bytes
// would end inside them.
// tiles_m, tiles_n: of a matrix; out: where the first result goes.
constexpr OutForm out_form(bool int32, int64_t M, int64_t N, int tiles_m, int tiles_n,
    uint64_t out, int64_t blocks) {
  const int64_t tiles = (int64_t)tiles_m * tiles_n, bytes = M * N * 4;
  if (!int32 || N % 32 == 0 || out % 4 != 0 || blocks <= 256 ||
      bytes < 6 * 1024 * tiles || blocks / tiles * bytes > 48000000)
    return kOutDirect;
  if (tiles_n == 1)
    return kOutTile;
  return out % 16 == 0 && N % 4 == 0 ? kOutRows : kOutDirect;
}

// The pieces of `bytes` bytes of int32 results that lie one after the other from `skew`
// bytes behind a multiple of 16 on, as offsets from that multiple: aligned ones of 16
// bytes from `first` up to `last`, and single results in front and behind, one to a
// thread.
struct TilePieces {
  int skew, first, last, end;
};
constexpr TilePieces tile_pieces(int skew, int bytes) {
  return {skew, skew ? 16 : 0, (skew + bytes) & ~15, skew + bytes};
}
// The single result that thread `tid` writes: four threads in front, the next four
// behind; negative: none.
constexpr int tile_end(const TilePieces &p, int tid) {
  const int o = tid < 4 ? p.skew + tid * 4
                        : (p.last > p.first ? p.last : p.first) + (tid - 4) * 4;
  return tid < 8 && o < p.end && (tid >= 4 || o < p.first) ? o : -1;
}

} // namespace gemm
} // namespace om
