// Answers questions about the batched product's launch rules, one a line, for
// 256 CUs:
//   q8 DTYPE ROWS UNITS N  ->  small nj ksplit bytes bound-of-N
#include <cstdio>

#include "gq_gemm_plan.h"

int main() {
  int dtype, rows, units, n;
  while (std::scanf(" q8 %d %d %d %d", &dtype, &rows, &units, &n) == 4) {
    const gq::Q8Plan p = gq::q8_plan(dtype, rows, units, n, 256);
    std::printf("%d %d %d %zu %zu\n", p.small, p.nj, p.ksplit, gq::q8_bytes(p, rows, units, n).total(),
                gq::q8_bytes_bound(rows, units, n, 256));
  }
}
