// How far the tiled kernels' copies and loads reach, as plain functions of the
// sizes: the kernels take their offsets from them, and a host program can walk
// a whole launch through them.
//
// A buffer descriptor's bound covers the per-lane offset.  Whether it covers
// the scalar offset too is not something to rely on, so a scalar offset always
// names a place inside the buffer.
#pragma once

#include <cstdint>

#ifdef __HIP__
#define PARROT_EXTENT __host__ __device__ __forceinline__ constexpr
#else
#define PARROT_EXTENT inline constexpr
#endif

namespace parrot {

// attention_tiles.hip: byte offset in one kv head's K (or V) fragments, nblk
// blocks of `pieces` KB, of KB `piece` of the two blocks from `first` on (of
// `first` once more where the second is missing).
PARROT_EXTENT uint32_t stage_piece_offset(int first, int piece, int pieces, int nblk) {
  const int missing = first + 1 < nblk ? 0 : pieces;
  return static_cast<uint32_t>(first * pieces + piece - (piece >= pieces ? missing : 0)) * 1024u;
}

// attention.hip, strided K: byte offset of row `key` of a sequence of T rows,
// `stride` elements apart.
PARROT_EXTENT uint32_t key_row_offset(int key, int T, int stride) {
  return static_cast<uint32_t>(key < T ? key : T - 1) * static_cast<uint32_t>(stride) * 2u;
}

// proj.hip, many rows: byte offset in the packed weight (N columns, ksteps
// 32-wide k steps) of k step `step` of the 16-column group `group` of the block
// that starts at column col0.
PARROT_EXTENT uint32_t column_group_offset(int col0, int group, int N, int ksteps, int step) {
  const int at = col0 / 16 + group, last = N / 16 - 1;
  return static_cast<uint32_t>((at < last ? at : last) * ksteps + step) * 1024u;
}

// gemm.hip, persistent tiles: the segment row whose id row r of row tile
// `tile` (bm rows) takes.
PARROT_EXTENT int tile_source_row(int tile, int bm, int r, int rows) {
  const int s = tile * bm + r;
  return s < rows ? s : rows - 1;
}

}  // namespace parrot
