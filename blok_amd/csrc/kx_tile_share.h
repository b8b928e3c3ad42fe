// kx_tile_share.h -- which of the tiles of kx_gemm_tile.h a product takes, and how they are shared out over workgroups: host code
// on sizes alone, in plain C++.
#pragma once
#include <stddef.h>

namespace kxtile {

struct TileSize {
  int tokens, rows;
  constexpr long sums() const { return (long)tokens * rows; }  // floats that a part of it leaves behind
  constexpr long of(int t, int r) const { return (long)((t + tokens - 1) / tokens) * ((r + rows - 1) / rows); }
};
constexpr TileSize LARGE = {256, 256}, MEDIUM = {128, 128}, SINGLE = {64, 128};

// How a product's tiles are shared out: a workgroup each for the first `whole`, `parts` workgroups with a part of the columns each for
// every further one, so that no round leaves CUs idle.  The parts have the first ids: as they end, early and unevenly, whole tiles
// take their places, where behind the whole tiles two of these would share a CU beside an idle one.
struct Share {
  int whole, parts;
  int grid(int tiles) const { return whole + (tiles - whole) * parts; }
};

// The shortest of: every tile whole; those beyond whole rounds in at most 16 `parts`; all of them in parts.  time(whole, rest, p): of
// `whole` tiles whole, in whole rounds of `round` where there are others, and `rest` tiles in p parts.
template <class Time>
inline Share share(long tiles, int round, int most_parts, long room, int arrivals, Time time, double *best, int least_parts = 1) {
  Share s = {(int)tiles, 1};
  *best = least_parts > 1 ? 1e30 : time(tiles, 0, 1);
  for (long whole = tiles / round * round, i = 0; i < 2; whole = 0, ++i) {
    const long rest = tiles - whole;
    const int most = whole && most_parts > 16 ? 16 : most_parts;
    for (int p = least_parts > 2 ? least_parts : 2; p <= most && rest > 0 && rest <= arrivals && rest * p <= room; ++p) {
      const double t = time(whole, rest, p);
      if (t < *best) *best = t, s = {(int)whole, p};
    }
    if (whole == 0) break;
  }
  return s;
}

// Which tile, and how it is shared out, for one product of `tokens` x `rows` with `blocks` blocks of 64 columns.
// Where the medium tiles leave CUs idle they take parts, of at least 16 blocks.  Beyond that the tile is the one that is sooner whole, by
// estimates in us: a round of large tiles takes 12 + 1.6 per block on 256 CUs, of medium ones (two per CU) 4.5 + 1.09; a last round of
// medium tiles that is not full takes its share of that, but no less than half, the time of one per CU.  Measured against it (us, 32-bit
// results, large / medium): large tiles in 1.5 rounds, medium ones in 3: 1536 x 16384 x 1024 75 / 69, x 2048 127 / 116, x 4096 228 / 211,
// x 8192 453 / 434, x 16384 855 / 886; 2048 x 16384 x 2048 150 / 214, 2048 x 8448 x 2048 116 / 94, 2048 x 5120 x 2048 64 / 61, 2048 x 36864 x
// 7168 1026 / 1265, 2048 x 7168 x 8192 252 / 329, 952 x 7168 x 18432 455 / 353, 700 x 12288 x 16384 379 / 428, 1024 x 36864 x 4096 359 / 345.
// In parts: 300 x 2048 x 8192 71 alone, 32 in four, 100 x 2048 x 8192 73 and 29 in eight, 2048 x 384 x 7168 65 and 32 in four.
struct Choice {
  bool large;
  Share s;
};
inline Choice choose(int tokens, int rows, int blocks, size_t part_floats, int arrivals, int cus) {
  const long medium = MEDIUM.of(tokens, rows), large = LARGE.of(tokens, rows);
  if (medium <= cus) {
    long p = cus / medium;
    if (p > blocks / 16) p = blocks / 16;
    if ((size_t)p > part_floats / MEDIUM.sums() / medium) p = part_floats / MEDIUM.sums() / medium;
    return p < 2 || medium > arrivals ? Choice{false, {(int)medium, 1}} : Choice{false, {0, (int)p}};
  }
  const long full = medium / (2 * cus), rest = medium % (2 * cus);
  const double rounds = full == 0 ? 1.0 : full + (rest == 0 ? 0.0 : rest <= cus ? 0.5 : rest / (2.0 * cus));
  const bool large_whole = (large + cus - 1) / cus * (12 + 1.6 * blocks) < rounds * (4.5 + 1.09 * blocks);
  // In parts where that is clearly sooner, by closer estimates (fitted to 4 to 20 ways of sharing out each of 5900 products, 65 to 2048 x
  // 512 to 40000 x 1024 to 18560): a workgroup that leaves its sums behind, and has them read, costs the memory's time for them, 0.032 us a
  // medium and 0.07 a large one; a last medium round takes 0.44 of a full one up to a workgroup per CU.  They are off by a tenth: parts have to
  // gain 15 % of their own time, 12 % of the whole product's where the tile is another one.  Of those products 62 are then more than 3 %
  // slower than whole, one by 11 %; 1329 are 3 % faster or more, and on average they take 0.973 of the time.  (With the whole tiles' estimate and 6 +
  // 2.5 per part, 12 + 8 for large ones, 582 were slower, by up to 47 %: 965 x 6110 x 3904 66 whole, 84 in two parts each.)
  auto medium_rounds = [&](long n, bool parts) {
    const long f = n / (2 * cus), r = n % (2 * cus);
    if (f == 0 && !parts) return 0.78 + (r <= cus ? 0.0 : 0.22 * (r - cus) / cus);
    return f + (r == 0 ? 0.0 : r <= cus ? 0.44 : 0.44 + 0.56 * (r - cus) / cus);
  };
  auto shared = [&](bool with_large) {
    return [=](long whole, long n, int p) {
      const double round = with_large ? 10 + 1.63 * blocks : 4.3 + 1.22 * blocks;
      const double t = whole == 0 ? 0.0 : round * (with_large ? (double)((whole + cus - 1) / cus) : medium_rounds(whole, n > 0));
      if (n == 0) return t;
      const double own = with_large ? (n * p + cus - 1) / cus * 1.63 * blocks / p + 9 * p + 0.07 * n * p : medium_rounds(n * p, true) * 1.22 * blocks / p + 0.032 * n * p;
      return with_large == large_whole ? t + 1.15 * own : 1.12 * (t + own);
    };
  };
  const int most = blocks / 16 < 8 ? blocks / 16 : 8;
  double tm, tl;
  const Share sm = share(medium, 2 * cus, most, part_floats / MEDIUM.sums(), arrivals, shared(false), &tm);
  const Share sl = share(large, cus, most, part_floats / LARGE.sums(), arrivals, shared(true), &tl);
  // whole tiles only of the size that is sooner whole
  if (large_whole) return sm.parts > 1 && tm < tl ? Choice{false, sm} : Choice{true, sl};
  return sl.parts > 1 && tl < tm ? Choice{true, sl} : Choice{false, sm};
}

// For the 32-bit tile and blocks of 32 columns.
inline Share choose_single(int tokens, int rows, int blocks, size_t part_floats, int arrivals, int cus) {
  const long tiles = SINGLE.of(tokens, rows);
  auto rounds = [&](long n, int p) { return (n * p + cus - 1) / cus * (1.5 + 0.97 * blocks / p + (p > 1 ? 2.5 : 0.0)); };
  // Two rounds of parts in front of a single round of whole tiles end so unevenly that CUs are left with two of those beside idle
  // ones: 464 x 6396 x 1024, 400 tiles, is a seventh slower with the last 144 in three parts each than whole.  Over 1900 products of more
  // tiles than CUs, 5 to 1024 x 128 to 16000 x 512 to 16384, what is chosen takes 0.85 of the whole tiles' time on average and 1.07 at most.
  auto time = [&](long whole, long rest, int p) { return whole == cus && rest * p > cus ? 1e30 : rounds(whole, 1) + rounds(rest, p); };
  // where two workgroups per CU are not filled by whole tiles, never fewer parts than fill them: the sums are as much shorter, and in 32
  // bits nearer to the exact ones (two parts instead of four were 1 % sooner and 8 % further off over a model of four layers; 64 x 1024 x
  // 16384 in 16 parts instead of 64 65 % further off)
  const long room = part_floats / SINGLE.sums(), most = blocks / 8;
  long least = 2 * cus / tiles < most ? 2 * cus / tiles : most;
  if (least > room / tiles) least = room / tiles;
  double best;
  return share(tiles, cus, (int)most, room, arrivals, time, &best, tiles > arrivals ? 1 : (int)least);
}

}  // namespace kxtile
