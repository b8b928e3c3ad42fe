// Answers the rule for experts' products of blok_amd/csrc/kx_tile_share.h: lines "pairs experts rows_in blocks_in rows_out blocks_out cus" on stdin, 1 for large tiles.
#include <stdio.h>
#include "kx_tile_share.h"

int main() {
  long pairs;
  int experts, cus;
  kxtile::ExpertMatrix in, out;
  while (scanf("%ld %d %d %d %d %d %d", &pairs, &experts, &in.rows, &in.blocks, &out.rows, &out.blocks, &cus) == 7)
    printf("%d\n", kxtile::experts_in_large_tiles(pairs, experts, in, out, cus));
}
