// Answers blok_amd/csrc/kx_gemv_chunks.h: lines "rows tile_rows most slots" on stdin, tiles of a chunk out.
#include <stdio.h>
#include "kx_gemv_chunks.h"

int main() {
  int rows, tile_rows, most, slots;
  while (scanf("%d %d %d %d", &rows, &tile_rows, &most, &slots) == 4) printf("%d\n", kxgemv::chunk_tiles(rows, tile_rows, most, slots));
}
