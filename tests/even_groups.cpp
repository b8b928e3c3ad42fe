// Answers kxtile::even_groups of blok_amd/csrc/kx_tile_share.h: lines "rows cols groups parts room arrivals cus" on stdin, workgroups per part out.
#include <stdio.h>
#include "kx_tile_share.h"

int main() {
  int rows, cols, groups, parts, arrivals, cus;
  size_t room;
  while (scanf("%d %d %d %d %zu %d %d", &rows, &cols, &groups, &parts, &room, &arrivals, &cus) == 7) printf("%d\n", kxtile::even_groups(rows, cols, groups, parts, room, arrivals, cus));
}
