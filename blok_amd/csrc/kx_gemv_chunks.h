// kx_gemv_chunks.h -- how many tiles a chunk of a one-token GEMV has where its workgroups take several chunks each (kx_dense.hip): host code on sizes
// alone, in plain C++.
#pragma once

namespace kxgemv {

// `slots` workgroups run at once and take the chunks in turn, so the launch takes as many chunks' time as the workgroup with the most has.  A chunk's time
// is its tiles' and that of two thirds of one more for its sums and its end: without that, chunks of one tile come out evenest and take longest.  us as
// one tile, as chosen and as eight: 66000 x 1536 48.5, 34.5 (six tiles), 42.1; 160633 x 2560 200, 129 (eight), 129; 66000 x 2048 52.5, 43.7 (six),
// 48.8; 37190 x 3072 54.8, 39.9 (five), 42.6; 18432 x 7168 46.8, 42.1 (three), 53.1.
// most: tiles of a chunk where it is alone.
inline int chunk_tiles(int rows, int tile_rows, int most, int slots) {
  auto time = [&](int tiles) {
    const long chunks = (rows + (long)tile_rows * tiles - 1) / ((long)tile_rows * tiles);
    return (chunks + slots - 1) / slots * (3 * tiles + 2);
  };
  int best = most;
  for (int tiles = most - 1; tiles >= 1; --tiles)
    if (time(tiles) < time(best)) best = tiles;
  return best;
}

}  // namespace kxgemv
