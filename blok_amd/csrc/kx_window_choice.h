// kx_window_choice.h -- whether a step of several positions attends in 32 bits on the matrix cores or in parts (kx_window.hip): host code on
// sizes alone, in plain C++.
#pragma once

namespace kxwin {

constexpr int GQ = 32;  // queries of a workgroup on the matrix cores

struct Step {
  int heads, kv_heads, columns;  // of a key and a value together, in the cache
  int batch, positions;
};
struct Split {
  int keys, parts;  // keys of a part; parts of the keys
  long at_once;     // tokens whose parts the scratch holds
};

// The sooner one by estimates in us, which leave out what both take.  On the matrix cores a workgroup of 32 queries and one head has a CU, and goes
// over all keys, in as many rounds as that makes.  Parts are launches of as many tokens as the scratch holds, each with a chain of a workgroup's keys
// for all query heads of a key head, rounds of workgroups, and the stream of the keys.  Fitted to 3200 steps of 2 to 900 positions of 1 to 64
// sequences behind up to 8000, windows of 64 and more, 2 to 64 heads of 32 to 256 columns with 1 to 16 to a key head: what is chosen takes 1.002 of the
// sooner one's time, 25 of them more than a tenth longer, 1.41 at most (an estimate by tokens and heads alone: 1.05, 477 and 4.0).  Whole operator, 8
// heads of 128 on 2 key heads (us, parts / matrix cores): 8 positions 15 / 24, 33 43 / 31, 100 93 / 33, with a window of 1024 777 316 / 75; 16 sequences of
// 50 558 / 35, 32 of 4 behind 200 26 / 37; 32 heads on 8, 20 positions behind 500 32 / 56.
// most, mean: keys of the last position, and on average.
inline bool matrix_cores_f32(const Step &s, int most, double mean, const Split &p, int cus) {
  const long groups = (long)s.heads * s.batch * ((s.positions + GQ - 1) / GQ), tokens = (long)s.batch * s.positions, rounds = (groups + cus - 1) / cus;
  const long at_once = p.at_once > 0 ? p.at_once : 1, launches = (tokens + at_once - 1) / at_once;
  const double columns = s.columns / 256.0, heads = s.heads / s.kv_heads, chain = (most < p.keys ? most : p.keys) / 64.0;
  const double cores = 1.05 * (8.2 + 15.1 * rounds * columns + 7.3 * ((rounds - 1) * mean + most) / 128 * columns);
  const double parts = 6.7 + launches * (6.8 + 0.75 * heads * columns + chain * (0.44 + 0.17 * heads * columns)) + (double)tokens * s.kv_heads * p.parts / cus * (1.6 + 0.4 * heads) +
                       tokens * columns * (66e-6 * mean * s.kv_heads + 78e-6 * (s.heads + 2 * s.kv_heads));
  return cores < parts;
}

}  // namespace kxwin
