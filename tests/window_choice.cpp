// Answers blok_amd/csrc/kx_window_choice.h: lines "heads kv_heads columns batch positions most mean keys parts at_once cus" on stdin, 1 for the matrix cores.
#include <stdio.h>
#include "kx_window_choice.h"

int main() {
  kxwin::Step s;
  kxwin::Split p;
  int most, cus;
  double mean;
  while (scanf("%d %d %d %d %d %d %lf %d %d %ld %d", &s.heads, &s.kv_heads, &s.columns, &s.batch, &s.positions, &most, &mean, &p.keys, &p.parts, &p.at_once, &cus) == 11)
    printf("%d\n", kxwin::matrix_cores_f32(s, most, mean, p, cus));
}
