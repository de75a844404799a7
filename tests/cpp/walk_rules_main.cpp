// Host-side checks of the walk's size rules (hbtplus_amd/csrc/hbt_walk_rules.hpp):
//  - every tree sent to a walk that stands at 32-bit byte offsets keeps all of
//    them below 2^32, from the root to the item after the sentinel;
//  - larger ones, up to the longest list the library takes, go to 64 lanes by
//    their segment and never to a launch's uniform group or to shared chunks,
//    under every tuning;
//  - targets whose potentials are summed in the reference's order (REPLAY) are
//    walked by each lane alone, at any numbers of sources and targets.
// Prints "ok" and exits 0, or names the first failed check and exits 1.
#include <cstdio>
#include <initializer_list>

#include "../../hbtplus_amd/csrc/hbt_walk_rules.hpp"

#define CHECK(cond, ...)                 \
  do {                                   \
    if (!(cond)) {                       \
      fprintf(stderr, "FAIL: ");         \
      fprintf(stderr, __VA_ARGS__);      \
      fprintf(stderr, "\n");             \
      return 1;                          \
    }                                    \
  } while (0)

using namespace hbt;

static int check_walk_forms() {
  const int64_t edge = (int64_t)1 << 26;
  const int64_t sizes[] = {1, 64, 1024, 420000, 46000000, edge - 2, edge - 1, edge, edge + 1, (int64_t)92 << 20, ((int64_t)1 << 30) - 2};
  const hbt_tuning tunings[] = {{{16, 16, 16}, {0, 1 << 30}, 2, 0, 64}, {{8, 8, 8}, {0, 1 << 30}, 2, 0, 16},
                                {{32, 32, 32}, {100, 700}, 2, 1, 1},    {{64, 64, 64}, {0, 1 << 30}, 2, 0, 64},
                                {{8, 16, 32}, {200, 3000}, 2, 0, 16},   {{64, 8, 16}, {200, 1 << 30}, 2, 0, 16}};
  for (const int64_t n : sizes)
    for (const hbt_tuning &t : tunings) {
      // pre-order positions 0 .. 2 n - 2, the sentinel, one item beyond it
      const bool reach = 32 * (2 * n + 1) <= (int64_t)1 << 32;
      const int own = walk_group_for(t, n), all = launch_group(t, n);
      CHECK(own == 8 || own == 16 || own == 32 || own == 64, "group %d of %lld", own, (long long)n);
      CHECK(reach || own == 64, "%lld sources walked at byte offsets by %d lanes", (long long)n, own);
      CHECK(reach || all == 0, "%lld sources walked by a launch's %d lanes", (long long)n, all);
      CHECK(all == 0 || all == own, "launch group %d, segment's %d (%lld)", all, own, (long long)n);
      // byte offsets are given up only at the end of their range
      CHECK(byte_walk(n) || n >= edge - 1, "%lld sources not walked at byte offsets", (long long)n);
      for (const int cus : {1, 32, 256, 304})
        CHECK(reach || walk_parts((n + 63) / 64, cus) == 1, "%lld sources' own walk shared", (long long)n);
    }
  return 0;
}

static int check_target_walks() {
  for (int64_t src = 1; src < (int64_t)1 << 30; src += 1 + src / 3)
    for (int64_t tgt = 1; tgt < (int64_t)1 << 34; tgt += 1 + tgt / 3)
      CHECK(target_walk(src, tgt, HBT_PREC_REPLAY) != TargetWalk::together, "REPLAY, %lld sources, %lld targets",
            (long long)src, (long long)tgt);
  return 0;
}

int main() {
  if (check_walk_forms() || check_target_walks()) return 1;
  printf("ok\n");
  return 0;
}
