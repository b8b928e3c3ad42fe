// Answers blok_amd/csrc/kx_read_once.h: lines "latent BYTES 0", "layers MODEL 0", "matrix BYTES MODEL" and "experts BYTES MODEL" on stdin, 1 for nontemporal copies
// and 0 for plain ones out.
#include <stdio.h>
#include <string>
#include "kx_read_once.h"

int main() {
  char what[16];
  size_t bytes, model;
  while (scanf("%15s %zu %zu", what, &bytes, &model) == 3) {
    const std::string w = what;
    printf("%d\n", w == "latent" ? kxonce::latent(bytes) : w == "layers" ? kxonce::layers(bytes) : w == "matrix" ? kxonce::matrix(bytes, model) : kxonce::experts(bytes, model));
  }
}
