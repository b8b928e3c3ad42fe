// Answers the rules of blok_amd/csrc/kx_tile_share.h: lines "f32 tokens rows blocks floats arrivals cus" on stdin, "large whole parts tiles twin" out.
#include <stdio.h>
#include "kx_tile_share.h"

int main() {
  int f32, tokens, rows, blocks, arrivals, cus;
  size_t floats;
  while (scanf("%d %d %d %d %zu %d %d", &f32, &tokens, &rows, &blocks, &floats, &arrivals, &cus) == 7) {
    kxtile::Choice c = {false, {0, 1}};
    if (f32) c.s = kxtile::choose_single(tokens, rows, blocks, floats, arrivals, cus);
    else c = kxtile::choose(tokens, rows, blocks, floats, arrivals, cus);
    printf("%d %d %d %ld %d\n", c.large, c.s.whole, c.s.parts, (f32 ? kxtile::SINGLE : c.large ? kxtile::LARGE : kxtile::MEDIUM).of(tokens, rows), c.twin);
  }
}
