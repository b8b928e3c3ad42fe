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

// Whole tiles of a product of `blocks` blocks of 64 columns, without what a launch takes: a last round costs most of a full one.
inline double large_rounds(double n, int blocks, int cus) {
  const long f = (long)(n / cus);
  const double r = n - (double)f * cus;
  return f * (13.8 + 1.45 * blocks) + (r == 0 ? 0.0 : 14.8 + (0.92 + 0.53 * r / cus) * blocks);
}
inline double medium_rounds(double n, int blocks, int cus) {  // two per CU
  const double round = 4.3 + (1.0 + 0.0009 * blocks) * blocks, lone = 2.2 + 0.463 * blocks;
  const long f = (long)(n / (2 * cus));
  const double r = n - 2.0 * f * cus;
  return f * round + (r == 0 ? 0.0 : r <= cus ? lone : lone + (round - lone) * (0.59 + 0.28 * (r - cus) / cus));  // a CU with two of the last round
}

// Which tile, and how it is shared out, for one product of `tokens` x `rows` with `blocks` blocks of 64 columns, by estimates in us that
// are fitted to measurements of 22000 products (65 to 2048 x 384 to 40000 x 256 to 18560, 32-bit results).
// Where the medium tiles leave CUs idle each has a CU to itself, in at least 10 blocks as the twin tile (kx_gemm_turns.h; at 4 blocks
// it takes 8 % longer than the medium one, at 10 2 % less, at 16 7 % and at 40 19 % less), and they take parts, of at least 16
// blocks: as many as fill the CUs, or more rounds of shorter ones where that is 5 % sooner (149 x 8548 x 18304, 134 tiles: 153 us whole, 103 in
// three).  300 x 2048 x 8192 53 alone, 28 in five, 100 x 2048 x 8192 52 and 28 in eight, 2048 x 384 x 7168 48 and 29 in five (as medium tiles alone 71, 73 and 65).
// Beyond that the tile is the one that is sooner whole, or in parts where that is clearly sooner: what is chosen takes 0.976 of the
// time of the sooner of whole medium and large tiles over 7000 products, 200 of them more than 3 % longer, and 1.5 % more than the best of
// every way to share out.  Measured (us, large / medium, whole): 2048 x 16384 x 2048 115 / 147, 2048 x 7168 x 8192 171 / 262, 2048 x 8192 x
// 2048 58 / 78, 2048 x 4096 x 2048 45 / 40, 1989 x 22265 x 1152 160 / 123, 945 x 32877 x 320 46 / 30; 260 x 11856 x 11904, 279 medium tiles,
// 196 whole, 116 as twin tiles with the last 23 in six parts.
struct Choice {
  bool large;
  Share s;
  bool twin = false;  // of the tiles of 128 x 128 those with two groups of waves
};
inline Choice choose(int tokens, int rows, int blocks, size_t part_floats, int arrivals, int cus) {
  const long medium = MEDIUM.of(tokens, rows), large = LARGE.of(tokens, rows);
  // n workgroups of `per` blocks: rounds of `round` + `block` per block, a last one of `last` and between `lone` and `block`
  auto rounds = [&](long n, double per, double round, double block, double last, double lone) {
    const long r = n % cus;
    return n / cus * (round + block * per) + (r == 0 ? 0.0 : last + (lone + (block - lone) * r / cus) * per);
  };
  if (medium <= cus) {
    const long room = medium > arrivals ? 0 : (long)(part_floats / MEDIUM.sums() / medium), most = room < blocks / 16 ? room : blocks / 16;
    auto time = [&](long p) { return 3.3 + rounds(medium * p, (double)blocks / p, 6.0, 0.458, 4.4, 0.327) + (p > 1 ? 0.9 + 1.4 * p + 0.009 * medium * p : 0.0); };
    long p = cus / medium < most ? cus / medium : most;
    if (p < 1) p = 1;
    const long fill = p;
    for (long q = fill + 1; q <= most && medium * q <= 4 * cus; ++q)
      if (time(q) * 1.05 < time(fill) && time(q) < time(p)) p = q;
    return {false, p == 1 ? Share{(int)medium, 1} : Share{0, (int)p}, blocks >= 10 * p};
  }
  auto whole_large = [&](long n) { return 3.3 + large_rounds(n, blocks, cus); };
  auto whole_medium = [&](long n) { return 5.5 + medium_rounds(n, blocks, cus); };
  const bool large_whole = whole_large(large) < whole_medium(medium);
  // In parts, or in rounds of twin tiles with the last one in parts: a workgroup that leaves its sums behind, and has them read,
  // costs the memory's time for them, 0.009 us a twin, 0.032 a medium and 0.074 a large one.  The estimates are off by a tenth: parts have to gain 15 %
  // of their own time, large ones 12 % of the product's where whole ones would be medium; twin tiles 22 % (with 12 % 48
  // of 1192 products in parts took more than a tenth longer than whole, now 5 of 960), 5 % where they are whole.
  const int most = blocks / 16 < 8 ? blocks / 16 : 8;
  auto large_time = [&](long n0, long n, int p) {
    const double t = n0 == 0 ? 0.0 : whole_large(n0);
    if (n == 0) return t;
    const double own = rounds(n * p, (double)blocks / p, 21.0, 1.36, 20.5, 0.63) + 0.8 * p + 0.074 * n * p;
    return large_whole ? t + 1.15 * own : 1.12 * (t + own);
  };
  auto medium_time = [&](long n0, long n, int p) {  // a last round takes 0.44 of a full one up to a workgroup per CU
    const double t = n0 == 0 ? 0.0 : whole_medium(n0);
    const long wgs = n * p, f = wgs / (2 * cus), r = wgs % (2 * cus);
    return n == 0 ? t : t + 1.15 * ((f + (r == 0 ? 0.0 : r <= cus ? 0.44 : 0.44 + 0.56 * (r - cus) / cus)) * (1.2 + 0.0009 * blocks) * blocks / p + 0.032 * wgs);
  };
  auto twin_time = [&](long n0, long n, int p) {
    const double t = n0 == 0 ? 0.0 : 3.3 + rounds(n0, blocks, 6.0, 0.458, 4.4, 0.327);
    return n == 0 ? 1.05 * t : 1.22 * (t + rounds(n * p, (double)blocks / p, 6.0, 0.458, 4.4, 0.327) + 0.9 + 1.4 * p + 0.009 * n * p);
  };
  double tm, tl, tt;
  const Share sm = share(medium, 2 * cus, most, part_floats / MEDIUM.sums(), arrivals, medium_time, &tm);
  const Share sl = share(large, cus, most, part_floats / LARGE.sums(), arrivals, large_time, &tl);
  const Share st = share(medium, cus, most, part_floats / MEDIUM.sums(), arrivals, twin_time, &tt);
  // whole large and medium tiles only of the size that is sooner whole
  if (!large_whole && sl.parts == 1) tl = 1e30;
  if (large_whole && sm.parts == 1) tm = 1e30;
  return tt < tl && tt < tm ? Choice{false, st, true} : tl < tm ? Choice{true, sl} : Choice{false, sm};
}

// Experts' products in large tiles, whose last one of an expert is computed in quarters, or in medium ones: `pairs` of tokens and experts
// meet two matrices of every expert.  How the pairs are spread is known on the device alone: even but for remainders.  A tile
// that is a quarter full takes 0.51 of a full one.  Large ones where they take less than 1.4 of the medium ones' estimate and 15 us a product behind
// it.  The operator over 1050 steps of 33 to 8192 tokens, 4 to 1000 experts of 3 x 256 to 7168 x 32 to 3000, spread evenly, unevenly and
// among 4 or 12 of them: what is chosen takes 1.003 of the sooner one's time and 25 of them are more than 3 % longer than in medium tiles
// or by the rule before (a large tile each for every expert fills the chip a fourth over: 1.040), by 14 % at most.  us, medium / large: 8 of 64 of 3 x
// 2048 x 1024, 2046 tokens 514 / 470, all among 8 222 / 191, 1024 tokens unevenly 350 / 372; 6 of 384 of 3 x 512 x 32, 8192 tokens 220 / 251; 2 of 16 of
// 3 x 7168 x 2048, 8192 tokens 2344 / 1918; 2 of 8 of 3 x 4096 x 1536, 1536 tokens 299 / 257.
struct ExpertMatrix {
  int rows, blocks;
};
inline bool experts_in_large_tiles(long pairs, int experts, ExpertMatrix in, ExpertMatrix out, int cus) {
  auto tiles = [&](int slots) { const double n = (double)pairs / slots + 0.3 * experts; return n > experts ? n : (double)experts; };
  const double full = 0.35 + 0.65 * tiles(64) / 4 / tiles(256);
  auto large = [&](ExpertMatrix m) { return 15.0 + full * large_rounds(tiles(256) * ((m.rows + 255) / 256), m.blocks, cus); };
  auto medium = [&](ExpertMatrix m) { return medium_rounds(tiles(128) * ((m.rows + 127) / 128), m.blocks, cus); };
  return large(in) + large(out) < 1.4 * (medium(in) + medium(out));
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

// Workgroups, each with all tokens (5 to 64), an equal share of the rows and one of `parts` parts of the columns, for a product whose rows make `groups` groups of
// 64: as many as fill whole rounds of one per CU.  Groups of 64 rows leave CUs with one beside others with two, or with none.  us, groups of 64 / shares:
// 17472 x 2048, 5 tokens 22.2 / 18.7 (273 to 512), 64 tokens 30.9 / 28.1; 9344 x 2048, 64 tokens 16.1 / 15.1 (146 to 256); 40000 x 2048 38.7 / 37.4 and 50.3 /
// 50.0 (625 to 768); 11003 x 2048 in two parts, 32 tokens 17.4 / 15.6 (344 to 512).  A workgroup copies 64 rows' places whatever its share is, so more
// rounds than that take longer, also where a CU holds two (up to 32 tokens): 40000 x 1024 as 1024 workgroups 23.3 at 32 tokens and 35.9 at 64, 20.9 and
// 30.2 as 768; 33000 x 2048 52.6 and 46.2.  The columns' parts, and with them the sums, stay as they are.
// Not for matrices for less than half of the CUs, nor for parts of less than 1024 columns, where starts and ends of the workgroups count for more than
// their rows (9344 x 2048 in three parts 12.2 and 12.3; models of 1024 columns 1 % longer).
// room: workgroups whose sums the scratch of the parts holds; arrivals: counters of groups.
inline int even_groups(int rows, int cols, int groups, int parts, size_t room, int arrivals, int cus) {
  const long all = (long)groups * parts;
  if (2 * all <= cus || cols < 1024 * parts) return groups;
  const long even = (all + cus - 1) / cus * cus / parts, n = even < rows ? even : rows;
  return n <= groups || n > arrivals || (size_t)(n * parts) > room ? groups : (int)n;
}

}  // namespace kxtile
