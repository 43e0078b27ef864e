"""Every offset that the tiled kernels' copies and loads take lies inside the
buffer it is taken in: the kernels' own index functions, compiled for the host
and walked through whole launches."""
import subprocess
from pathlib import Path

KERNELS = Path(__file__).resolve().parent.parent / "parrot-h200-worker_amd" / "parrot" / "kernels"


def _run(tmp_path, body):
    source, program = tmp_path / "walk.cpp", tmp_path / "walk"
    source.write_text('#include "extents.h"\n#include <algorithm>\n#include <cstdio>\n'
                      "using namespace parrot;\nint main() {\n" + body + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{KERNELS}", str(source), "-o",
                    str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


def test_attention_stages_stay_inside_the_fragments(tmp_path):
    """Every sequence length over several blocks, windows inside a block and
    longer than the sequence, every query tile, both blocks of each stage."""
    _run(tmp_path, """
  for (int d : {64, 96, 128})
    for (int T = 1; T <= 330; ++T)
      for (int W : {1, 33, 77, 4096})
        for (int rows : {32, 64, 128})  // queries per workgroup
          for (int wg0 = 0; wg0 < T; wg0 += rows) {
            const int nblk = (T + 31) / 32, pieces = d / 16;
            const long bytes = static_cast<long>(nblk) * 32 * d * 2;
            const int lo = std::max(0, wg0 - W + 1) / 32;
            const int stages = ((std::min(wg0 + rows, T) - 1) / 32 - lo) / 2 + 1;
            for (int st = 0; st < stages; ++st)
              for (int piece = 0; piece < 2 * pieces; ++piece) {
                const long at = stage_piece_offset(lo + 2 * st, piece, pieces, nblk);
                const int block = lo + 2 * st + piece / pieces;
                const long want = (static_cast<long>(std::min(block, nblk - 1)) * pieces + piece % pieces) * 1024;
                if (at + 1024 > bytes || at != want) {
                  std::printf("d=%d T=%d W=%d wg0=%d stage %d piece %d: %ld of %ld\\n", d, T, W, wg0,
                              st, piece, at, bytes);
                  return 1;
                }
              }
          }
  return 0;""")


def test_projection_columns_stay_inside_the_weight(tmp_path):
    """Every width up to 1600 columns, also as two ranges of blocks (keys, then
    values): each block of 48 columns, whole or with groups past the last."""
    _run(tmp_path, """
  for (int ksteps : {4, 8, 16, 24})
    for (int N = 16; N <= 1600; N += 16)
      for (int n_swap : {0, N / 2 / 16 * 16, N}) {
        const long bytes = static_cast<long>(N) * ksteps * 64;
        const int first = (n_swap + 47) / 48, total = first + (N - n_swap + 47) / 48;
        for (int blk = 0; blk < total; ++blk)
          for (int j = 0; j < 3; ++j)
            for (int step = 0; step < ksteps; ++step) {
              const int col0 = blk < first ? blk * 48 : n_swap + (blk - first) * 48;
              const long at = column_group_offset(col0, j, N, ksteps, step);
              const long want = (static_cast<long>(std::min(col0 / 16 + j, N / 16 - 1)) * ksteps + step) * 1024;
              if (at + 1024 > bytes || at != want) {
                std::printf("N=%d n_swap=%d block %d group %d step %d: %ld of %ld\\n", N, n_swap, blk, j,
                            step, at, bytes);
                return 1;
              }
            }
      }
  return 0;""")


def test_strided_key_rows_stay_inside_the_sequence(tmp_path):
    """Every 32-key block of every sequence length, packed and padded rows."""
    _run(tmp_path, """
  for (int d : {64, 96, 128})
    for (int stride : {d, 8 * d + 8})
      for (int T = 1; T <= 300; ++T)
        for (int k0 = 0; k0 < T; k0 += 32)
          for (int key = k0; key < k0 + 32; ++key) {
            const long at = key_row_offset(key, T, stride);
            const long want = static_cast<long>(std::min(key, T - 1)) * stride * 2;
            if (at != want || at + d * 2 > (static_cast<long>(T - 1) * stride + d) * 2) {
              std::printf("d=%d stride=%d T=%d key %d: %ld\\n", d, stride, T, key, at);
              return 1;
            }
          }
  return 0;""")


def test_every_row_of_an_expert_tile_takes_a_row_of_its_segment(tmp_path):
    """Every segment length, whole tiles and partial last ones: no row of a
    tile is left without an id of the segment."""
    _run(tmp_path, """
  for (int rows = 1; rows <= 700; ++rows)
    for (int tile = 0; tile * 128 < rows; ++tile)
      for (int r = 0; r < 128; ++r) {
        const int s = tile_source_row(tile, 128, r, rows);
        if (s != std::min(tile * 128 + r, rows - 1)) {
          std::printf("rows=%d tile %d row %d: %d\\n", rows, tile, r, s);
          return 1;
        }
      }
  return 0;""")
