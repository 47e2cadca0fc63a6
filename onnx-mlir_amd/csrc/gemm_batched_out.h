// How results leave k_gemm_i8_batched (gemm_batched.hip): the choice and the pieces
// that a tile is written in, as functions of sizes and addresses alone, which run on
// host and device.
#pragma once

#include <cstdint>

namespace om {
namespace gemm {

enum OutForm : int { kOutDirect, kOutTile, kOutRows };

// By way of LDS where rows are no whole lines and the grid is more than one round of
// blocks: up to that the barrier and the second way cost more than the stores (48 x
// 38x38x80 4.74 us by LDS, 4.57 without).
//   Tiles as wide as the matrix: 156 x 82x128x82 7.6 -> 6.8 us, 64 x 511x511x64 with 8-bit
//   results 13.9 -> 9.6, the loads' part of both included.
//   Rows of whole 16-byte pieces: int32 88 x 472x128x472 28.8 -> 23.4; not 8-bit ones (21.2
//   -> 23.5), nor other rows, whose ends are stores of their own (64 x 511x64x511 17.2
//   -> 18.5).
// result: bytes of one; out: where the first goes.  Results that do not start on a
// multiple of their size are stored one by one: pieces of 16 bytes would end inside
// them.
constexpr OutForm out_form(int result, int N, int tiles_n, uint64_t out, int64_t blocks) {
  if (blocks <= 256 || (int64_t)N * result % 128 == 0 || out % (uint64_t)result != 0)
    return kOutDirect;
  if (tiles_n == 1)
    return kOutTile;
  return result == 4 && out % 16 == 0 && N % 4 == 0 ? kOutRows : kOutDirect;
}

// The pieces of `bytes` bytes of results that lie one after the other from `skew`
// bytes behind a multiple of 16 on, as offsets from that multiple: aligned ones of 16
// bytes from `first` up to `last`, and single results in front and behind, one to a
// thread.
struct TilePieces {
  int skew, first, last, end;
};
constexpr TilePieces tile_pieces(int skew, int bytes) {
  return {skew, skew ? 16 : 0, (skew + bytes) & ~15, skew + bytes};
}
// The single result of ES bytes that thread `tid` writes: 16 / ES threads in front,
// the next 16 / ES behind; negative: none.
template <int ES>
constexpr int tile_end(const TilePieces &p, int tid) {
  constexpr int PER = 16 / ES;
  const int o = tid < PER ? p.skew + tid * ES
                          : (p.last > p.first ? p.last : p.first) + (tid - PER) * ES;
  return tid < 2 * PER && o < p.end && (tid >= PER || o < p.first) ? o : -1;
}

} // namespace gemm
} // namespace om
