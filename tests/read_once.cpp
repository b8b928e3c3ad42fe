// Answers blok_amd/csrc/kx_read_once.h: lines "latent BYTES" on stdin, 1 for nontemporal copies and 0 for plain ones out.
#include <stdio.h>
#include <string.h>
#include "kx_read_once.h"

int main() {
  char what[16];
  size_t bytes;
  while (scanf("%15s %zu", what, &bytes) == 2) printf("%d\n", kxonce::latent(bytes));
}
