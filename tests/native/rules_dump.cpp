// Dispatch rules of csrc/layout.hpp, for tests/test_rules.py: one query per input line.
//   tiles S ntiles C K width f64    -> post_level_tiles
//   tau ntiles C tiles_per_chunk    -> tau_chunk_tiles
//   dwalk S C I levels ntiles K     -> use_dwalk
//   route S C I levels ntiles K dense split -> use_dwalk
//   nat S C split post ntiles dense -> use_nat_rows
#include <cstdio>
#include <cstring>

#include "layout.hpp"

int main() {
  char what[16];
  while (std::scanf("%15s", what) == 1) {
    if (!std::strcmp(what, "tiles")) {
      int S, nt, C, K, w, f;
      if (std::scanf("%d %d %d %d %d %d", &S, &nt, &C, &K, &w, &f) != 6) return 1;
      std::printf("%d\n", hx::post_level_tiles(nt, S, C, K, w, f != 0));
    } else if (!std::strcmp(what, "tau")) {
      int nt, C, t;
      if (std::scanf("%d %d %d", &nt, &C, &t) != 3) return 1;
      std::printf("%d\n", hx::tau_chunk_tiles(nt, C, t));
    } else if (!std::strcmp(what, "dwalk")) {
      int S, C, I, h, nt, K;
      if (std::scanf("%d %d %d %d %d %d", &S, &C, &I, &h, &nt, &K) != 6) return 1;
      std::printf("%d\n", (int)hx::use_dwalk(S, C, I, h, nt, K));
    } else if (!std::strcmp(what, "route")) {
      int S, C, I, h, nt, K, d, f;
      if (std::scanf("%d %d %d %d %d %d %d %d", &S, &C, &I, &h, &nt, &K, &d, &f) != 8) return 1;
      std::printf("%d\n", (int)hx::use_dwalk(S, C, I, h, nt, K, d != 0, f != 0));
    } else if (!std::strcmp(what, "nat")) {
      int S, C, f, post, nt, d;
      if (std::scanf("%d %d %d %d %d %d", &S, &C, &f, &post, &nt, &d) != 6) return 1;
      std::printf("%d\n", (int)hx::use_nat_rows(S, C, f != 0, post != 0, nt, d != 0));
    } else {
      return 1;
    }
  }
  return 0;
}
