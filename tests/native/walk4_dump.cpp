// Reads T and (T-1) post-order triples on stdin, prints the programs of the four-state FP32 walks
// as the plan builds them (hx::build_post4, hx::build_pre4): the exponent stack's size, then one
// line of 4 ints per post-order entry and one line of 8 ints per pre-order entry. Host-only test
// driver.
#include <cstdio>
#include <vector>

#include "walk.hpp"

int main() {
  int T = 0;
  if (std::scanf("%d", &T) != 1 || T < 2) return 2;
  const int I = T - 1, nn = 2 * T - 1;
  std::vector<int32_t> post(3 * I), kids(2 * nn, -1);
  for (int r = 0; r < I; ++r) {
    if (std::scanf("%d %d %d", &post[3 * r], &post[3 * r + 1], &post[3 * r + 2]) != 3) return 2;
    kids[2 * post[3 * r]] = post[3 * r + 1];
    kids[2 * post[3 * r] + 1] = post[3 * r + 2];
  }
  std::vector<int32_t> walk, segtab, cher, cher_row, post4, pre, pre4;
  std::vector<uint8_t> drop, drop4;
  int need = 0, slots = 0, depth = 0;
  if (!hx::build_walk(T, kids, post.data(), walk, segtab, need, &drop)) return 1;
  hx::list_cherries(T, kids, post.data(), cher, cher_row);
  if (!hx::build_post4(T, walk, post4, slots, drop4)) return 1;
  if (!hx::build_pre_walk(T, kids, post.data(), pre, depth, &drop4, &cher_row)) return 1;
  if (!hx::build_pre4(T, pre, drop4, pre4)) return 1;
  std::printf("%d %d\n", slots, need);
  for (int i = 0; i < I; ++i)
    for (int q = 0; q < 4; ++q)
      std::printf("%d%c", post4[(size_t)hx::kPost4Ints * i + q], q < 3 ? ' ' : '\n');
  for (int i = 0; i < I; ++i)
    for (int q = 0; q < 8; ++q)
      std::printf("%d%c", pre4[(size_t)hx::kPre4Ints * i + q], q < 7 ? ' ' : '\n');
  return 0;
}
