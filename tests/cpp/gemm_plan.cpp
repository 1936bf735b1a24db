// Answers questions about the batched product's launch rules, one a line, for
// 256 CUs:
//   q8 DTYPE ROWS UNITS N               ->  small nj ksplit bytes bound-of-N
//   quad DTYPE ROWS UNITS N             ->  ksplit of the short-batch bf16 kernel,
//                                           and whether a batch takes that kernel
//   room N                              ->  tokens that workspace is taken for
//   take HELD DENIED NEED ROOM LIMIT    ->  ok held denied allocations, where at
//                                           most LIMIT bytes are to be had
#include <cstdio>
#include <cstring>

#include "gq_gemm_plan.h"

int main() {
  char what[8];
  int dtype, rows, units, n;
  while (std::scanf("%7s", what) == 1) {
    if (!std::strcmp(what, "q8") && std::scanf("%d %d %d %d", &dtype, &rows, &units, &n) == 4) {
      const gq::Q8Plan p = gq::q8_plan(dtype, rows, units, n, 256);
      std::printf("%d %d %d %zu %zu\n", p.small, p.nj, p.ksplit, gq::q8_bytes(p, rows, units, n).total(),
                  gq::q8_bytes_bound(rows, units, n, 256));
    } else if (!std::strcmp(what, "quad") && std::scanf("%d %d %d %d", &dtype, &rows, &units, &n) == 4) {
      const int tiles = (rows + gq::GEMM_QUAD_ROWS - 1) / gq::GEMM_QUAD_ROWS;
      std::printf("%d %d\n", gq::gemm_quad_ksplit(dtype, tiles, rows, units, n, 256),
                  gq::gemm_quad_faster(dtype, rows, units, n, 256));
    } else if (!std::strcmp(what, "room") && std::scanf("%d", &n) == 1) {
      std::printf("%ld\n", gq::gemm_room_tokens(n));
    } else if (!std::strcmp(what, "take")) {
      size_t held, denied, need, room, limit;
      if (std::scanf("%zu %zu %zu %zu %zu", &held, &denied, &need, &room, &limit) != 5) return 1;
      char own = 0, fresh = 0;
      void *p = held ? &own : nullptr;
      int calls = 0;
      const bool ok = gq::take_workspace(p, held, denied, need, room, [&](size_t b) -> void * {
        calls++;
        return b <= limit ? &fresh : nullptr;
      });
      if (ok && p == nullptr) return 1;
      std::printf("%d %zu %zu %d\n", ok, held, denied, calls);
    } else {
      return 1;
    }
  }
}
